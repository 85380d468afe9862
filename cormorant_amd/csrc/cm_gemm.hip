// cm_gemm.hip -- exact int16 x int16 contractions on CDNA4 i8 MFMA: the Matmul unit and
// the standard (group 1) Conv unit as an implicit GEMM; the depthwise conv runs direct.
//
// Arithmetic.  Every int16 operand x is written x - 128 = 256 h + l with h = x >> 8 and
// l = (x & 255) - 128, both signed bytes (the low byte with its top bit flipped).  Then
//   sum_k a b = sum_k A'B' + 128 sum_k a + 128 sum_k b - 16384 K,   A' = a - 128, B' = b - 128
//   sum_k A'B' = 2^16 HH + 2^8 (HL + LH) + LL
// where HH, HL, LH, LL are sums of byte products, each exact in int32 (|h l| <= 2^14, so
// K <= 32768 keeps HL + LH below 2^31).  Per 32 x 32 block and 32-k substep, four
// v_mfma_i32_32x32x32_i8 accumulate HH, MID = HL + LH and LL; the epilogue recombines them
// with the row / column sums in int32 (int64 only for K > 8192 on the saturating path) and
// applies the unit's output rule: floor(acc / 2^8) saturated to int16, after an int32 wrap
// for the power-of-two path.  Padding of k (beyond K or past the channels of a conv tile)
// is the byte pair (0, 0) -- A' = 0 -- on both sides and is left out of the sums, so it
// contributes nothing.
//
// Data flow: split kernels write the two byte planes of A as [rows][kp] and of B as
// [cols][kp] (k contiguous, the MFMA operand order; B transposed in registers or LDS), plus
// per-1024-k partial row / column sums; the plane GEMM streams 64-k tiles of the four planes
// into LDS with direct global -> LDS copies and sums the partials in its prologue.
#include "cm_common.h"
#include "cm_rowops_math.h"

#include <type_traits>

namespace cm {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));

constexpr int BN = 128, BK = 64;               // output tile columns; k step in elements (= plane bytes)
constexpr int SLAB = 1024;                     // k per partial-sum slab

// Where batch slice bt of an operand starts: (bt / inner) s1 + (bt % inner) s2 elements (the
// (sequence, head) pairs of an attention's operands inside one projection), or bt s1.
struct Slices {
    uint64_t s1 = 0, s2 = 0;
    uint32_t inner = 1;
    __host__ __device__ uint64_t off(uint32_t bt) const {
        return inner > 1 ? (uint64_t)(bt / inner) * s1 + (uint64_t)(bt % inner) * s2 : (uint64_t)bt * s1;
    }
};

__device__ __forceinline__ uint32_t pack_hi(const int16_t* v) {   // 4 high bytes
    return (uint32_t)(uint8_t)(v[0] >> 8) | ((uint32_t)(uint8_t)(v[1] >> 8) << 8) |
           ((uint32_t)(uint8_t)(v[2] >> 8) << 16) | ((uint32_t)(uint8_t)(v[3] >> 8) << 24);
}
__device__ __forceinline__ uint32_t pack_lo(const int16_t* v) {   // 4 low bytes, top bit flipped
    return ((uint32_t)(uint8_t)v[0] | ((uint32_t)(uint8_t)v[1] << 8) |
            ((uint32_t)(uint8_t)v[2] << 16) | ((uint32_t)(uint8_t)v[3] << 24)) ^ 0x80808080u;
}

// ---------------------------------------------------------------- operand sources
// B side: columns of the output; B(kk, j) of the GEMV image of more than one column group (the other
// matmul images have their own kernels).
struct SrcGemvB {
    const int16_t* p;
    uint32_t k, m, kw;
    __device__ bool real(uint32_t j, uint32_t kk) const { return j < m && kk < k; }
    __device__ int16_t at(uint32_t j, uint32_t kk) const {
        uint32_t c = (kk / (16 * kw)) * 16 + (kk & 15), jj = (kk >> 4) % kw;
        return p[((uint64_t)c * m + j) * kw + jj];
    }
};
// Conv weights in the packed tile-major layout (ConvKernel.h:136-159) as GEMM rows:
// kk = ((ict * kh + khi) * kw + kwi) * 16 + lane; lanes past in_ch are padding.
struct SrcConvW {
    const int16_t* p;
    uint32_t out_ch, in_ch, kh, kw, tiles, per_m, last_lanes;
    __device__ bool real(uint32_t mo, uint32_t kk) const {
        uint32_t lane = kk & 15, t = kk >> 4, ict = t / (kh * kw);
        return mo < out_ch && ict < tiles && ict * 16 + lane < in_ch;
    }
    __device__ int16_t at(uint32_t mo, uint32_t kk) const {
        uint32_t lane = kk & 15, t = kk >> 4, ict = t / (kh * kw), pos = t - ict * kh * kw;
        uint32_t lanes = ict + 1 == tiles ? last_lanes : 16;
        return p[(uint64_t)mo * per_m + (uint64_t)ict * kh * kw * 16 + pos * lanes + lane];
    }
};
// im2col of one NCHW image as GEMM columns: column p = oh * out_w + ow.
struct Im2col {
    const int16_t* p;
    uint64_t img;                    // elements per image
    uint32_t in_ch, in_h, in_w, out_w, kh, kw, sh, sw, dh, dw, pt, pl, cols;
};

// Split one operand into byte planes [lines][kp] (lines = rows for A, columns for B) and
// partial line sums per SLAB of k.  Workgroup: 64 lines x one SLAB; the 64x64 element tiles
// pass through LDS so that the reads follow the source's fast dimension (`KFast`: k for conv
// weights; the line index for B images).
template <class Src, bool KFast>
__global__ __launch_bounds__(256) void split_kernel(Src src, uint64_t src_slice, int8_t* __restrict__ hi,
                                                    int8_t* __restrict__ lo, int32_t* __restrict__ part,
                                                    uint32_t lines_p, uint32_t kp, uint32_t nslab) {
    __shared__ int16_t tile[64][64 + 2];
    __shared__ uint8_t realt[64][64 + 4];
    const uint32_t l0 = blockIdx.x * 64, slab = blockIdx.y, bt = blockIdx.z;
    Src s = src;
    s.p = src.p + bt * src_slice;
    const uint64_t pl = (uint64_t)bt * lines_p * kp;
    const uint32_t t = threadIdx.x;
    const uint32_t my_line = t >> 2, part_k = (t & 3) * 16;
    int32_t sum = 0;
    const uint32_t k_end = min(kp, (slab + 1) * SLAB);
    for (uint32_t k0 = slab * SLAB; k0 < k_end; k0 += 64) {
        for (uint32_t r = 0; r < 16; r++) {
            uint32_t idx = r * 256 + t, a, b;
            if (KFast) { a = idx >> 6; b = idx & 63; }       // a = line, b = k
            else { b = idx >> 6; a = idx & 63; }             // b = k, a = line
            bool re = s.real(l0 + a, k0 + b);
            tile[a][b] = re ? s.at(l0 + a, k0 + b) : (int16_t)0;
            realt[a][b] = re;
        }
        __syncthreads();
        int16_t v[16];
        uint32_t hw[4], lw[4];
        for (int q = 0; q < 16; q++) {
            v[q] = tile[my_line][part_k + q];
            if (realt[my_line][part_k + q]) sum += v[q];
        }
        for (int q = 0; q < 4; q++) {
            hw[q] = pack_hi(v + 4 * q);
            lw[q] = pack_lo(v + 4 * q);
            // padding is the byte pair (0, 0)
            for (int e = 0; e < 4; e++)
                if (!realt[my_line][part_k + 4 * q + e]) {
                    hw[q] &= ~(0xFFu << (8 * e));
                    lw[q] &= ~(0xFFu << (8 * e));
                }
        }
        const uint64_t off = pl + (uint64_t)(l0 + my_line) * kp + k0 + part_k;
        *reinterpret_cast<uint4*>(hi + off) = make_uint4(hw[0], hw[1], hw[2], hw[3]);
        *reinterpret_cast<uint4*>(lo + off) = make_uint4(lw[0], lw[1], lw[2], lw[3]);
        __syncthreads();
    }
    sum += __shfl_xor(sum, 1, 64);
    sum += __shfl_xor(sum, 2, 64);
    if ((t & 3) == 0) part[((uint64_t)bt * nslab + slab) * lines_p + l0 + my_line] = sum;
}

// ---------------------------------------------------------------- bandwidth split kernels
// Padding is written as the value 128 (A' = 0: the byte pair (0, 0)) and left out of the sums.
constexpr int16_t kPad = 128;

// 8 elements at any element alignment (one 16-byte load: global loads need no more than 2 bytes).
__device__ __forceinline__ int4 load8(const int16_t* p) {
    int4 v;
    __builtin_memcpy(&v, p, 16);
    return v;
}

// All of the wave's loads have arrived.  Before the first store of a split whose loads stand in branches:
// each later group of values would else be waited for together with the stores of the groups before it
// (packed 4096 x 4096: split_cols_kernel 16.8 us without, 16.0 with; 2048 rows of 4096: split_rows_kernel 8.75, 8.27).
__device__ __forceinline__ void loads_landed() { __builtin_amdgcn_s_waitcnt(0x0F70); }

// Rows with k contiguous (the matmul A, row stride lda, rows at any alignment): one wavefront
// per row and SLAB of k, 8 k per lane per 16-byte load, the slab's loads all in flight
// before the first is used; only the lane at the end of a row loads single elements.  Rows of 771
// (3000 of them) took 59 us through the general kernel's 2-byte loads, 8.5 here.
// Grid (ceil(lines_p / 4), nslab, slices).
__global__ __launch_bounds__(256) void split_rows_kernel(const int16_t* __restrict__ src, Slices slice,
                                                         uint64_t lda, uint32_t rows, uint32_t k,
                                                         int8_t* __restrict__ hi, int8_t* __restrict__ lo,
                                                         int32_t* __restrict__ part, uint32_t lines_p,
                                                         uint32_t kp, uint32_t nslab) {
    constexpr int U = SLAB / 512;
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t row = blockIdx.x * 4 + (threadIdx.x >> 6), slab = blockIdx.y, bt = blockIdx.z;
    if (row >= lines_p) return;
    const int16_t* r = src + slice.off(bt) + (uint64_t)row * lda;
    const uint64_t po = ((uint64_t)bt * lines_p + row) * kp;
    const bool real_row = row < rows;
    int4 v[U];
    if (real_row && (slab + 1) * SLAB <= k) {          // the whole slab is real: no branches
#pragma unroll
        for (int u = 0; u < U; u++) v[u] = load8(r + slab * SLAB + 512 * u + 8 * lane);
    } else {
#pragma unroll
        for (int u = 0; u < U; u++) {
            const uint32_t k0 = slab * SLAB + 512 * u + 8 * lane;
            if (real_row && k0 + 8 <= k) {
                v[u] = load8(r + k0);
                continue;
            }
            int16_t e[8];
#pragma unroll
            for (int q = 0; q < 8; q++) e[q] = (real_row && k0 + q < k) ? r[k0 + q] : kPad;
            v[u] = *reinterpret_cast<const int4*>(e);
        }
    }
    loads_landed();
    int32_t sum = 0;
#pragma unroll
    for (int u = 0; u < U; u++) {
        const uint32_t k0 = slab * SLAB + 512 * u + 8 * lane;
        if (k0 >= kp) continue;
        if (real_row && k0 + 8 <= k) {
            sum += sum8(v[u]);
        } else {
            const int16_t* e = reinterpret_cast<const int16_t*>(&v[u]);
#pragma unroll
            for (int q = 0; q < 8; q++)
                if (real_row && k0 + q < k) sum += e[q];
        }
        uint2 h, l;
        split8(v[u], h, l);
        *reinterpret_cast<uint2*>(hi + po + k0) = h;
        *reinterpret_cast<uint2*>(lo + po + k0) = l;
    }
    for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 64);
    if (lane == 0) part[((uint64_t)bt * nslab + slab) * lines_p + row] = sum;
}

// Rows of at most 256 k (kp in {64, 128, 192, 256}: one slab): G lanes per row (kp / 8, and 32
// for kp 192 with the last 8 idle), one 16-byte load each, 64 / G rows per wavefront, the row
// sum over the row's lane group.
// Grid (ceil(lines_p / (4 * 64 / G)), 1, slices).
template <uint32_t G>
__global__ __launch_bounds__(256) void split_rows_short_kernel(const int16_t* __restrict__ src, Slices slice,
                                                               uint64_t lda, uint32_t rows, uint32_t k,
                                                               int8_t* __restrict__ hi, int8_t* __restrict__ lo,
                                                               int32_t* __restrict__ part, uint32_t lines_p,
                                                               uint32_t kp) {
    constexpr uint32_t RPW = 64 / G;                       // rows per wavefront
    const uint32_t lane = threadIdx.x & 63, g = lane % G;
    const uint32_t row = (blockIdx.x * 4 + (threadIdx.x >> 6)) * RPW + lane / G, bt = blockIdx.z;
    const uint32_t k0 = 8 * g;
    const bool in = row < lines_p && k0 < kp, real_row = row < rows;
    int4 v = make_int4(0, 0, 0, 0);
    int32_t sum = 0;
    if (in) {
        const int16_t* r = src + slice.off(bt) + (uint64_t)row * lda;
        if (real_row && k0 + 8 <= k) {
            v = load8(r + k0);
            sum = sum8(v);
        } else {
            int16_t e[8];
#pragma unroll
            for (int q = 0; q < 8; q++) {
                const bool re = real_row && k0 + q < k;
                e[q] = re ? r[k0 + q] : kPad;
                sum += re ? e[q] : 0;
            }
            v = *reinterpret_cast<const int4*>(e);
        }
    }
#pragma unroll
    for (uint32_t off = 1; off < G; off <<= 1) sum += __shfl_xor(sum, off, 64);
    if (!in) return;
    uint2 h, l;
    split8(v, h, l);
    const uint64_t po = ((uint64_t)bt * lines_p + row) * kp + k0;
    *reinterpret_cast<uint2*>(hi + po) = h;
    *reinterpret_cast<uint2*>(lo + po) = l;
    if (g == 0) part[(uint64_t)bt * lines_p + row] = sum;
}

// Columns of a k-major image (row-major B [k][m] at any width and alignment, or the packed
// 32-column tiles; 771 x 1235 71 us through the general kernel, 11 here).  A wavefront takes 32 columns and 256 k of one SLAB: lane = (r4, c8) with
// r4 = lane / 4 picking 4 consecutive k of each 64-k group and c8 = lane % 4 picking 8
// columns, so one load instruction reads 16 rows x 64 contiguous bytes.  Each lane loads
// its 4 groups x 4 rows x 8 columns at once, then transposes every 4 x 8 block in registers
// (byte permutes) into one dword of 4 k per column and plane.  A workgroup is the four
// 256-k quarters of one slab; their column sums meet in LDS.  Grid (ceil(lines_p / 32),
// nslab, slices).
__global__ __launch_bounds__(256) void split_cols_kernel(const int16_t* __restrict__ src, Slices slice,
                                                         uint64_t ldb, uint32_t packed, uint32_t m, uint32_t k,
                                                         int8_t* __restrict__ hi, int8_t* __restrict__ lo,
                                                         int32_t* __restrict__ part, uint32_t lines_p,
                                                         uint32_t kp, uint32_t nslab) {
    __shared__ int32_t csum[4][32];
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t r4 = lane >> 2, c8 = lane & 3;
    const uint32_t jg = blockIdx.x * 32, slab = blockIdx.y, bt = blockIdx.z;
    const uint32_t j0 = jg + 8 * c8;                       // this lane's first column
    const int16_t* b = src + slice.off(bt);
    const uint32_t kq = slab * SLAB + 256 * wave;          // this wave's first k
    const bool cols_real = j0 + 8 <= m;
    // element (kk, j) of the image
    auto at = [&](uint32_t kk, uint32_t j) -> uint64_t {
        return packed ? ((uint64_t)(j >> 5) * k + kk) * 32 + (j & 31) : (uint64_t)kk * ldb + j;
    };
    int4 v[4][4];
    if (cols_real && kq + 256 <= k) {                  // every load is real: no branches
        const int16_t* p0 = b + at(kq + 4 * r4, j0);
        const uint64_t rs = packed ? 32 : ldb;         // elements per k row
#pragma unroll
        for (int g = 0; g < 4; g++)
#pragma unroll
            for (int r = 0; r < 4; r++) v[g][r] = load8(p0 + (64 * g + r) * rs);
    } else if (cols_real || packed || m >= 8) {
        // whole loads for the real k rows.  The lane at the last columns: a packed tile holds all its
        // 32 columns, and the ones past m become padding; of row-major rows it loads the last 8 and
        // shifts out the ones its left neighbour holds.  The lanes past m hold padding alone.
        const uint32_t nv = cols_real ? 8 : (j0 < m ? m - j0 : 0);           // real columns
        const uint32_t jl = cols_real || packed ? j0 : m - 8;
        const int4 pad = make_int4(0x00800080, 0x00800080, 0x00800080, 0x00800080);
#pragma unroll
        for (int g = 0; g < 4; g++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const uint32_t kk = kq + 64 * g + 4 * r4 + r;
                v[g][r] = pad;
                if (kk < k && nv) v[g][r] = load8(b + at(kk, jl));
            }
        if (nv && nv < 8) {
            const unsigned __int128 mask = ((unsigned __int128)1 << (16 * nv)) - 1;
            const uint32_t sh = packed ? 0 : 16 * (8 - nv);
            unsigned __int128 fill;
            __builtin_memcpy(&fill, &pad, 16);
#pragma unroll
            for (int g = 0; g < 4; g++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    unsigned __int128 w;
                    __builtin_memcpy(&w, &v[g][r], 16);
                    w = ((w >> sh) & mask) | (fill & ~mask);
                    if (kq + 64 * g + 4 * r4 + r < k) __builtin_memcpy(&v[g][r], &w, 16);
                }
        }
    } else {
#pragma unroll
        for (int g = 0; g < 4; g++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const uint32_t kk = kq + 64 * g + 4 * r4 + r;
                int16_t e[8];
#pragma unroll
                for (int q = 0; q < 8; q++) e[q] = (kk < k && j0 + q < m) ? b[at(kk, j0 + q)] : kPad;
                v[g][r] = *reinterpret_cast<const int4*>(e);
            }
    }
    loads_landed();
    int32_t sum[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int g = 0; g < 4; g++) {
        const uint32_t k0 = kq + 64 * g + 4 * r4;
        if (k0 >= kp) continue;
        uint32_t d[4][4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            d[r][0] = (uint32_t)v[g][r].x; d[r][1] = (uint32_t)v[g][r].y;
            d[r][2] = (uint32_t)v[g][r].z; d[r][3] = (uint32_t)v[g][r].w;
            if (k0 + r < k) {
                const int16_t* e = reinterpret_cast<const int16_t*>(&v[g][r]);
#pragma unroll
                for (int q = 0; q < 8; q++)
                    if (j0 + q < m) sum[q] += e[q];
            }
        }
#pragma unroll
        for (int c2 = 0; c2 < 4; c2++) {               // columns 2 c2 and 2 c2 + 1
            const uint32_t xh = __builtin_amdgcn_perm(d[1][c2], d[0][c2], 0x07030501u);
            const uint32_t yh = __builtin_amdgcn_perm(d[3][c2], d[2][c2], 0x07030501u);
            const uint32_t xl = __builtin_amdgcn_perm(d[1][c2], d[0][c2], 0x06020400u);
            const uint32_t yl = __builtin_amdgcn_perm(d[3][c2], d[2][c2], 0x06020400u);
            const uint64_t o0 = ((uint64_t)bt * lines_p + j0 + 2 * c2) * kp + k0;
            const uint64_t o1 = o0 + kp;
            *reinterpret_cast<uint32_t*>(hi + o0) = __builtin_amdgcn_perm(yh, xh, 0x05040100u);
            *reinterpret_cast<uint32_t*>(hi + o1) = __builtin_amdgcn_perm(yh, xh, 0x07060302u);
            *reinterpret_cast<uint32_t*>(lo + o0) = __builtin_amdgcn_perm(yl, xl, 0x05040100u) ^ 0x80808080u;
            *reinterpret_cast<uint32_t*>(lo + o1) = __builtin_amdgcn_perm(yl, xl, 0x07060302u) ^ 0x80808080u;
        }
    }
    // column sums: over the 16 lanes of one c8 (lane bits 2..5), then the four waves
#pragma unroll
    for (int q = 0; q < 8; q++) {
        int32_t x = sum[q];
        for (int off = 4; off < 64; off <<= 1) x += __shfl_xor(x, off, 64);
        sum[q] = x;
    }
    if (r4 == 0) {
#pragma unroll
        for (int q = 0; q < 8; q++) csum[wave][8 * c8 + q] = sum[q];
    }
    __syncthreads();
    if (threadIdx.x < 32 && jg + threadIdx.x < lines_p)
        part[((uint64_t)bt * nslab + slab) * lines_p + jg + threadIdx.x] =
            csum[0][threadIdx.x] + csum[1][threadIdx.x] + csum[2][threadIdx.x] + csum[3][threadIdx.x];
}

// 1x1 stride-1 convolutions with the images folded into the GEMM's columns: line
// j = img * plane + p is pixel p of image img, k the input channel, B(c, j) = x[img][c][p].
// For planes that are not a multiple of 8 pixels.  A workgroup takes 64 lines and one SLAB
// of k, each of its waves (up to 16) 64 k in 16-k chunks: lane = line, 16 loads of 2 bytes
// (the 64 lanes of one load read 128 consecutive bytes of one channel row where the lines
// stay in one image), packed into one 16-byte word per plane.  Grid (lines_p / 64, nslab).
__global__ __launch_bounds__(1024) void split_fold_kernel(const int16_t* __restrict__ x, uint32_t in_ch,
                                                          uint32_t plane, uint64_t img_elems, uint32_t cols,
                                                          int8_t* __restrict__ hi, int8_t* __restrict__ lo,
                                                          int32_t* __restrict__ part, uint32_t lines_p, uint32_t kp) {
    __shared__ int32_t wsum[16][64];
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
    const uint32_t j = blockIdx.x * 64 + lane, slab = blockIdx.y;
    const bool real = j < cols;
    const uint32_t img = real ? j / plane : 0, p = real ? j - img * plane : 0;
    const int16_t* src = x + img * img_elems + p;
    int32_t sum = 0;
    const uint32_t kb = slab * SLAB + 64 * wave, ke = min(kb + 64, kp);
    // the wave's four 16-k chunks unrolled: every load in flight before the first is used
#pragma unroll 4
    for (uint32_t k0 = kb; k0 < ke; k0 += 16) {
        int16_t e[16];
        if (real && k0 + 16 <= in_ch) {
#pragma unroll
            for (int q = 0; q < 16; q++) e[q] = src[(uint64_t)(k0 + q) * plane];
#pragma unroll
            for (int q = 0; q < 16; q++) sum += e[q];
        } else {
#pragma unroll
            for (int q = 0; q < 16; q++) {
                const bool r = real && k0 + q < in_ch;
                e[q] = r ? src[(uint64_t)(k0 + q) * plane] : kPad;
                sum += r ? e[q] : 0;
            }
        }
        uint2 h0, l0, h1, l1;
        split8(*reinterpret_cast<const int4*>(e), h0, l0);
        split8(*reinterpret_cast<const int4*>(e + 8), h1, l1);
        const uint64_t off = (uint64_t)j * kp + k0;
        *reinterpret_cast<uint4*>(hi + off) = make_uint4(h0.x, h0.y, h1.x, h1.y);
        *reinterpret_cast<uint4*>(lo + off) = make_uint4(l0.x, l0.y, l1.x, l1.y);
    }
    wsum[wave][lane] = sum;
    __syncthreads();
    if (wave == 0) {
        int32_t t = 0;
        for (uint32_t w = 0; w < waves; w++) t += wsum[w][lane];
        part[(uint64_t)slab * lines_p + j] = t;
    }
}

// The same operand for few lines (small planes): 16 lines a workgroup so that the grid has
// four times the workgroups.  Wave w takes the slab's 64 k from 64 w; lane (line l % 16, chunk
// l / 16) loads its line's 16 k of the chunk (the 16 lanes of one chunk read 32 consecutive bytes
// of a channel row where the lines stay in one image), so the four chunk lanes of a line write
// 64 contiguous bytes of each plane.  Grid (lines_p / 16, nslab).
__global__ __launch_bounds__(1024) void split_fold16_kernel(const int16_t* __restrict__ x, uint32_t in_ch,
                                                            uint32_t plane, uint64_t img_elems, uint32_t cols,
                                                            int8_t* __restrict__ hi, int8_t* __restrict__ lo,
                                                            int32_t* __restrict__ part, uint32_t lines_p,
                                                            uint32_t kp) {
    __shared__ int32_t wsum[16][16];
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
    const uint32_t ln = lane & 15, ch = lane >> 4;
    const uint32_t j = blockIdx.x * 16 + ln, slab = blockIdx.y;
    const bool real = j < cols;
    const uint32_t img = real ? j / plane : 0, p = real ? j - img * plane : 0;
    const int16_t* src = x + img * img_elems + p;
    int32_t sum = 0;
    const uint32_t k0 = slab * SLAB + 64 * wave + 16 * ch;
    if (k0 < kp) {
        int16_t e[16];
        if (real && k0 + 16 <= in_ch) {
#pragma unroll
            for (int q = 0; q < 16; q++) e[q] = src[(uint64_t)(k0 + q) * plane];
#pragma unroll
            for (int q = 0; q < 16; q++) sum += e[q];
        } else {
#pragma unroll
            for (int q = 0; q < 16; q++) {
                const bool r = real && k0 + q < in_ch;
                e[q] = r ? src[(uint64_t)(k0 + q) * plane] : kPad;
                sum += r ? e[q] : 0;
            }
        }
        uint2 h0, l0, h1, l1;
        split8(*reinterpret_cast<const int4*>(e), h0, l0);
        split8(*reinterpret_cast<const int4*>(e + 8), h1, l1);
        const uint64_t off = (uint64_t)j * kp + k0;
        *reinterpret_cast<uint4*>(hi + off) = make_uint4(h0.x, h0.y, h1.x, h1.y);
        *reinterpret_cast<uint4*>(lo + off) = make_uint4(l0.x, l0.y, l1.x, l1.y);
    }
    sum += __shfl_xor(sum, 16, 64);
    sum += __shfl_xor(sum, 32, 64);
    if (ch == 0) wsum[wave][ln] = sum;
    __syncthreads();
    if (threadIdx.x < 16) {
        int32_t t = 0;
        for (uint32_t w = 0; w < waves; w++) t += wsum[w][threadIdx.x];
        part[(uint64_t)slab * lines_p + blockIdx.x * 16 + threadIdx.x] = t;
    }
}

// im2col planes of NCHW images, k in the packed weight order (16-channel tiles x kernel positions):
// as split_fold16_kernel, 16 columns (output pixels) a workgroup, wave w the slab's 64 k from 64 w;
// lane (column l % 16, chunk l / 16) loads its pixel's 16 channels at the chunk's kernel position
// (16 loads in flight, one address and one bounds test a chunk) and writes 16 bytes a plane, the
// four chunk lanes of a column 64 contiguous bytes.  Bound by the planes' bytes: 8 images of 64
// channels at 56 x 56, 3 x 3 (29 MB of planes) took 67 us with a division and bounds
// tests per element, 12.8 here.  Grid (lines_p / 16, nslab, images).
__global__ __launch_bounds__(1024) void split_im2col_kernel(Im2col g, int8_t* __restrict__ hi,
                                                            int8_t* __restrict__ lo, int32_t* __restrict__ part,
                                                            uint32_t lines_p, uint32_t kp, uint32_t nslab) {
    __shared__ int32_t wsum[16][16];
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
    const uint32_t ln = lane & 15, ch = lane >> 4;
    const uint32_t j = blockIdx.x * 16 + ln, slab = blockIdx.y, bt = blockIdx.z;
    const uint32_t k0 = slab * SLAB + 64 * wave + 16 * ch;
    int32_t sum = 0;
    if (k0 < kp) {
        const uint32_t t = k0 >> 4, khw = g.kh * g.kw, ict = t / khw, pos = t - ict * khw;
        const uint32_t khi = pos / g.kw, kwi = pos - khi * g.kw, c0 = ict * 16;
        const uint32_t oh = j / g.out_w, ow = j - oh * g.out_w;
        const int64_t ih = (int64_t)oh * g.sh + (int64_t)khi * g.dh - g.pt;
        const int64_t iw = (int64_t)ow * g.sw + (int64_t)kwi * g.dw - g.pl;
        const bool inside = ih >= 0 && ih < (int64_t)g.in_h && iw >= 0 && iw < (int64_t)g.in_w;
        const uint32_t nc = j < g.cols && c0 < g.in_ch ? min(g.in_ch - c0, 16u) : 0;     // real channels
        const uint64_t plane = (uint64_t)g.in_h * g.in_w;
        const int16_t* src = g.p + bt * g.img + (inside ? c0 * plane + (uint64_t)ih * g.in_w + (uint64_t)iw : 0);
        int16_t e[16];
        if (nc == 16 && inside) {
#pragma unroll
            for (int q = 0; q < 16; q++) e[q] = src[q * plane];
#pragma unroll
            for (int q = 0; q < 16; q++) sum += e[q];
        } else {
#pragma unroll
            for (int q = 0; q < 16; q++) {
                const bool r = (uint32_t)q < nc;
                e[q] = r ? (inside ? src[q * plane] : (int16_t)0) : kPad;
                sum += r ? e[q] : 0;
            }
        }
        uint2 h0, l0, h1, l1;
        split8(*reinterpret_cast<const int4*>(e), h0, l0);
        split8(*reinterpret_cast<const int4*>(e + 8), h1, l1);
        const uint64_t off = ((uint64_t)bt * lines_p + j) * kp + k0;
        *reinterpret_cast<uint4*>(hi + off) = make_uint4(h0.x, h0.y, h1.x, h1.y);
        *reinterpret_cast<uint4*>(lo + off) = make_uint4(l0.x, l0.y, l1.x, l1.y);
    }
    sum += __shfl_xor(sum, 16, 64);
    sum += __shfl_xor(sum, 32, 64);
    if (ch == 0) wsum[wave][ln] = sum;
    __syncthreads();
    if (threadIdx.x < 16) {
        int32_t t = 0;
        for (uint32_t w = 0; w < waves; w++) t += wsum[w][threadIdx.x];
        part[((uint64_t)bt * nslab + slab) * lines_p + blockIdx.x * 16 + threadIdx.x] = t;
    }
}

// The folded operand for planes with many lines: a workgroup takes 64 lines and one SLAB of
// k in 64 x 64 tiles through LDS.  Thread t loads line t % 64 at 16 k (2-byte loads, the 64
// lanes of one load on consecutive lines), then packs 16 consecutive k of line t / 4 into
// 16-byte words: the four threads of a line write 64 contiguous bytes of each plane.
// Grid (lines_p / 64, nslab).
__global__ __launch_bounds__(256) void split_fold_lds_kernel(const int16_t* __restrict__ x, uint32_t in_ch,
                                                             uint32_t plane, uint64_t img_elems, uint32_t cols,
                                                             int8_t* __restrict__ hi, int8_t* __restrict__ lo,
                                                             int32_t* __restrict__ part, uint32_t lines_p,
                                                             uint32_t kp) {
    __shared__ int16_t tile[64][64 + 2];
    const uint32_t t = threadIdx.x, la = t & 63, kr = t >> 6;
    const uint32_t l0 = blockIdx.x * 64, slab = blockIdx.y;
    const uint32_t ja = l0 + la;
    const bool real_a = ja < cols;
    const uint32_t img = real_a ? ja / plane : 0, pa = real_a ? ja - img * plane : 0;
    const int16_t* src = x + img * img_elems + pa;
    const uint32_t my_line = t >> 2, part_k = (t & 3) * 16;
    int32_t sum = 0;
    const uint32_t k_end = min(kp, (slab + 1) * SLAB);
    // a 64-k chunk's loads in registers, the next chunk's issued while this one is split
    int16_t v[16];
    auto load_chunk = [&](uint32_t k0) {
#pragma unroll
        for (uint32_t r = 0; r < 16; r++) {
            const uint32_t kk = k0 + 4 * r + kr;
            v[r] = (real_a && kk < in_ch) ? src[(uint64_t)kk * plane] : kPad;
        }
    };
    load_chunk(slab * SLAB);
    for (uint32_t k0 = slab * SLAB; k0 < k_end; k0 += 64) {
#pragma unroll
        for (uint32_t r = 0; r < 16; r++) tile[la][4 * r + kr] = v[r];
        __syncthreads();
        if (k0 + 64 < k_end) load_chunk(k0 + 64);
        int16_t e[16];
#pragma unroll
        for (int q = 0; q < 16; q++) {
            e[q] = tile[my_line][part_k + q];
            sum += (l0 + my_line < cols && k0 + part_k + q < in_ch) ? e[q] : 0;
        }
        uint2 h0, lw0, h1, lw1;
        split8(*reinterpret_cast<const int4*>(e), h0, lw0);
        split8(*reinterpret_cast<const int4*>(e + 8), h1, lw1);
        const uint64_t off = (uint64_t)(l0 + my_line) * kp + k0 + part_k;
        *reinterpret_cast<uint4*>(hi + off) = make_uint4(h0.x, h0.y, h1.x, h1.y);
        *reinterpret_cast<uint4*>(lo + off) = make_uint4(lw0.x, lw0.y, lw1.x, lw1.y);
        __syncthreads();
    }
    sum += __shfl_xor(sum, 1, 64);
    sum += __shfl_xor(sum, 2, 64);
    if ((t & 3) == 0) part[(uint64_t)slab * lines_p + l0 + my_line] = sum;
}

// ---------------------------------------------------------------- epilogues
// An epilogue names where output row `i` of slice `bt` starts (nullptr past the last row),
// the raw per-row bias (added to the sum as bias << 8), the offset of column `j` from a row
// start, and whether every row start and the column count are even (then two adjacent
// results go out as one 4-byte store).
struct TileBase {               // a tile's first output element and row stride (nullptr: none)
    int16_t* base;
    uint32_t ld;
};
struct EpiMatmul {              // C[bt][i][j] = c + off(bt) + i * ldc + j
    int16_t* c;
    uint64_t c_bs;
    uint32_t rows, cols, wrap, pairs;
    uint64_t ldc = 0;           // row stride (0: cols)
    uint64_t c_bs2 = 0;         // with `inner` > 1: slice bt at (bt / inner) c_bs + (bt % inner) c_bs2
    uint32_t inner = 1;
    int32_t lo = -32768, hi = 32767;    // output bounds (the saturation; a fused RELU / RELU6 narrows them)
    __device__ int32_t row_bias(uint32_t) const { return 0; }
    __device__ int16_t* row_ptr(uint32_t bt, uint32_t i) const {
        if (i >= rows) return nullptr;
        const uint64_t off = inner > 1 ? (uint64_t)(bt / inner) * c_bs + (uint64_t)(bt % inner) * c_bs2 : bt * c_bs;
        return c + off + (uint64_t)i * (ldc ? ldc : cols);
    }
    __device__ uint64_t col_off(uint32_t j) const { return j; }
    // The tile (row0, col0) of tm x tn wholly inside C with paired stores: its first element
    // and the row stride, so that element (r, c) of the tile sits at base + r * ld + c.
    __device__ __forceinline__ TileBase tile_base(uint32_t bt, uint32_t row0, uint32_t col0, uint32_t tm,
                                                  uint32_t tn) const {
        const uint64_t l = ldc ? ldc : cols;
        if (!pairs || row0 + tm > rows || col0 + tn > cols || l * tm >= (1ull << 30)) return TileBase{nullptr, 0};
        return TileBase{row_ptr(bt, row0) + col0, (uint32_t)l};
    }
};
struct EpiConv {                // y pattern (ConvKernel.h:250-258); acc seeded with bias << 8
    int16_t* y;
    const int16_t* bias;
    uint64_t img;               // elements per image (out_ch * plane)
    uint32_t rows, cols, cs, cn, gs, wrap, pairs;
    uint32_t fold;              // pixels per image when the images are folded into the columns, else 0
    int32_t lo = -32768, hi = 32767;    // output bounds (the saturation; a fused RELU / RELU6 narrows them)
    __device__ int32_t row_bias(uint32_t i) const { return bias && i < rows ? (int32_t)bias[i] : 0; }
    __device__ int16_t* row_ptr(uint32_t bt, uint32_t i) const {
        if (i >= rows) return nullptr;
        const uint64_t base = cn ? (uint64_t)(i % cn) * cs + (uint64_t)(i / cn) * gs : (uint64_t)i * cs;
        return y + bt * img + base;
    }
    __device__ uint64_t col_off(uint32_t j) const {
        if (!fold) return j;
        const uint32_t im = j / fold;
        return (uint64_t)im * img + (j - im * fold);
    }
    __device__ __forceinline__ TileBase tile_base(uint32_t bt, uint32_t row0, uint32_t col0, uint32_t tm,
                                                  uint32_t tn) const {
        if (!pairs || fold || cn || row0 + tm > rows || col0 + tn > cols || (uint64_t)cs * tm >= (1ull << 30))
            return TileBase{nullptr, 0};
        return TileBase{row_ptr(bt, row0) + col0, cs};
    }
};

// Recombination modes of the output rule floor(acc / 2^8) -> int16:
//   acc = 2^16 HH + 2^8 MID + LL + 128 rowsum + 128 colsum - 16384 K + 2^8 bias.
// With rowsum = 2 rh' + rl', colsum likewise (arithmetic shift, low bit),
//   floor(acc / 2^8) = 2^8 HH + MID + rh + ch + ((LL + rl + cl) >> 8),
//   rh = bias - 64 K + (rowsum >> 1), rl = 128 (rowsum & 1), ch = colsum >> 1, cl = 128 (colsum & 1),
// every term but 2^8 HH exact in int32 for K <= 32768.
//   kSatNarrow (K <= 8192): |the rest| < 2^29.1, so clamping HH to +-2^22 keeps the sum in
//     int32 and cannot change a saturated result (|2^8 HH| > 2^30 then decides the sign);
//   kWrap: the sum wrapped to int32 first, i.e. floor(acc / 2^8) mod 2^24, sign-extended;
//   kSatWide (K > 8192, saturating): the sum in int64.
//   kSplitFix (wrap products split over k): every slice stores its 2^16 HH + 2^8 MID + LL
//     mod 2^32 as int32 partials, and the slice of a tile that arrives last adds the others'
//     to its own and stores the tile by the kWrap rule (split_fixup).
enum : uint32_t { kSatNarrow = 0, kWrap = 1, kSatWide = 2, kSplitFix = 3 };

__device__ __forceinline__ int32_t clamp_i32(int32_t v, int32_t lo, int32_t hi) {   // v_med3_i32
    return min(max(v, lo), hi);
}

// The result is clamped to [lo, hi] inside the int16 range: the saturation, or with a fused
// RELU (lo = 0) / RELU6 (lo = 0, hi = 6 * 2^8) the activation of the saturated value as well.
template <uint32_t MODE>
__device__ __forceinline__ int32_t recombine(int32_t hh, int32_t mid, int32_t ll, int32_t rhch, int32_t rlcl,
                                             int32_t lo, int32_t hi) {
    const int32_t y = mid + rhch + ((ll + rlcl) >> 8);
    int32_t q;
    if (MODE == kSatNarrow) {
        q = (int32_t)((uint32_t)clamp_i32(hh, -(1 << 22), 1 << 22) << 8) + y;
    } else if (MODE == kWrap) {
        q = (int32_t)(((uint32_t)hh << 8) + (uint32_t)y);
        q = (q << 8) >> 8;
    } else {
        const long long w = ((long long)hh << 8) + (long long)mid + (long long)rhch + ((ll + rlcl) >> 8);
        q = (int32_t)(w > 32767 ? 32767 : (w < -32768 ? -32768 : w));
    }
    return clamp_i32(q, lo, hi);
}

typedef int v16i __attribute__((ext_vector_type(16)));

// Store one wave's (32 RB) x (32 CB) results.  A lane holds D[8 (r / 4) + 4 lh + r % 4][l32] of
// each 32 x 32 block.  With PAIRS, lanes 2c and 2c + 1 swap one result per row pair (DPP
// quad_perm [1,0,3,2]) so that the even lane stores columns (2c, 2c + 1) of row r and the
// odd lane the same columns of row r + 1, as one 4-byte store each.
template <uint32_t MODE, bool PAIRS, int RB, int CB, class Epi>
__device__ __forceinline__ void store_wave_tile(const v16i (&hh)[RB][CB], const v16i (&mid)[RB][CB],
                                                const v16i (&ll)[RB][CB], const int2* rterm, const int2* cterm,
                                                uint32_t bt, uint32_t row0, uint32_t col0, uint32_t wr,
                                                uint32_t wc, uint32_t l32, uint32_t lh, const Epi& epi) {
    const uint32_t odd = l32 & 1;
#pragma unroll
    for (int j = 0; j < CB; j++) {
        const uint32_t cl = wc * (32 * CB) + j * 32 + l32, col = col0 + cl;
        const int2 ct = cterm[cl];
#pragma unroll
        for (int i = 0; i < RB; i++) {
#pragma unroll
            for (int r = 0; r < 16; r += 2) {
                const uint32_t rl = wr * (32 * RB) + i * 32 + 8 * (r >> 2) + 4 * lh + (r & 3);
                const int2 r0 = rterm[rl], r1 = rterm[rl + 1];
                const int32_t q0 = recombine<MODE>(hh[i][j][r], mid[i][j][r], ll[i][j][r], r0.x + ct.x, r0.y + ct.y,
                                                   epi.lo, epi.hi);
                const int32_t q1 = recombine<MODE>(hh[i][j][r + 1], mid[i][j][r + 1], ll[i][j][r + 1], r1.x + ct.x,
                                                   r1.y + ct.y, epi.lo, epi.hi);
                if (PAIRS) {
                    const int32_t give = odd ? q0 : q1;
                    const int32_t got = __builtin_amdgcn_mov_dpp(give, 0xB1, 0xF, 0xF, false);
                    const uint32_t lo = (uint32_t)(odd ? got : q0) & 0xFFFFu;
                    const uint32_t hi = (uint32_t)(odd ? q1 : got) << 16;
                    int16_t* dst = epi.row_ptr(bt, row0 + rl + odd);
                    if (dst != nullptr && col - odd < epi.cols)
                        *reinterpret_cast<uint32_t*>(dst + epi.col_off(col - odd)) = lo | hi;
                } else if (col < epi.cols) {
                    int16_t* d0 = epi.row_ptr(bt, row0 + rl);
                    int16_t* d1 = epi.row_ptr(bt, row0 + rl + 1);
                    const uint64_t co = epi.col_off(col);
                    if (d0 != nullptr) d0[co] = (int16_t)q0;
                    if (d1 != nullptr) d1[co] = (int16_t)q1;
                }
                // one row pair at a time: hoisting the term loads of later pairs would
                // need more registers than the accumulators leave
                if constexpr (RB * CB >= 4) __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
}

// store_wave_tile for a tile wholly inside the output with plain rows (tile_base): the lane's
// offset from the tile's first element in 32 bits, the row offsets uniform, no bounds checks.
template <uint32_t MODE, int RB, int CB>
__device__ __forceinline__ void store_wave_fast(const v16i (&hh)[RB][CB], const v16i (&mid)[RB][CB],
                                                const v16i (&ll)[RB][CB], const int2* rterm, const int2* cterm,
                                                int16_t* __restrict__ base, uint32_t ld, uint32_t wr, uint32_t wc,
                                                uint32_t l32, uint32_t lh, int32_t lo, int32_t hi) {
    const uint32_t odd = l32 & 1;
    const uint32_t lane_off = (wr * (32 * RB) + 4 * lh + odd) * ld + wc * (32 * CB) + l32 - odd;
#pragma unroll
    for (int j = 0; j < CB; j++) {
        const int2 ct = cterm[wc * (32 * CB) + j * 32 + l32];
#pragma unroll
        for (int i = 0; i < RB; i++) {
#pragma unroll
            for (int r = 0; r < 16; r += 2) {
                const uint32_t rl = wr * (32 * RB) + i * 32 + 8 * (r >> 2) + 4 * lh + (r & 3);
                const int2 r0 = rterm[rl], r1 = rterm[rl + 1];
                const int32_t q0 = recombine<MODE>(hh[i][j][r], mid[i][j][r], ll[i][j][r], r0.x + ct.x, r0.y + ct.y,
                                                   lo, hi);
                const int32_t q1 = recombine<MODE>(hh[i][j][r + 1], mid[i][j][r + 1], ll[i][j][r + 1], r1.x + ct.x,
                                                   r1.y + ct.y, lo, hi);
                // the pair exchange of store_wave_tile: the even lane stores row r, the odd lane row r + 1
                const int32_t give = odd ? q0 : q1;
                const int32_t got = __builtin_amdgcn_mov_dpp(give, 0xB1, 0xF, 0xF, false);
                const uint32_t lo = (uint32_t)(odd ? got : q0), hi = (uint32_t)(odd ? q1 : got);
                const uint32_t roff = (uint32_t)(i * 32 + 8 * (r >> 2) + (r & 3)) * ld + j * 32;
                *reinterpret_cast<uint32_t*>(base + lane_off + roff) = __builtin_amdgcn_perm(hi, lo, 0x05040100u);
                if constexpr (RB * CB >= 4) __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
}

// kSplitFix: this slice's partial of its wave's 64 x 64 outputs, in the accumulators' own
// layout (a tile's nz slices are consecutive blocks of NW RB CB KiB x 4 at `tile_part`, NW the
// workgroup's waves; in a block, wave w's accumulator (i, j) rows 4q .. 4q + 3 sit at 1 KiB row
// (4 (CB i + j) + q) of the wave's 4 RB CB KiB, 16 bytes a lane), written and read with agent-scope 16-byte buffer
// accesses (sc1) so that a workgroup on another XCD reads them; then the tile's arrival count.
// The slice that arrives last (ticket nz - 1) resets the count for the next launch, adds the
// other slices' partials (all were stored, and their stores had completed, before their slices
// took their tickets) and returns true with the wrapped total T in limb form -- HH = T >> 16,
// MID = (T >> 8) & 255, LL = T & 255, 2^16 HH + 2^8 MID + LL = T exactly -- for the kWrap
// store; the other slices return false.  No workgroup waits for another.  Every wave of the
// workgroup calls it (two barriers).
template <int NW, int RB, int CB>
__device__ __forceinline__ bool split_fixup(v16i (&hh)[RB][CB], v16i (&mid)[RB][CB], v16i (&ll)[RB][CB],
                                            int32_t* tile_part, uint32_t nz, uint32_t kz, uint32_t wave,
                                            uint32_t lane, uint32_t* cnt, uint32_t* ticket) {
    constexpr uint32_t kWave = 4096 * RB * CB, kBlock = NW * kWave;   // bytes of one slice's wave, tile
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(tile_part, 0, (int)(nz * kBlock), 0x00020000);
    const uint32_t wbase = wave * kWave + lane * 16;
#pragma unroll
    for (int i = 0; i < RB; i++)
#pragma unroll
        for (int j = 0; j < CB; j++)
#pragma unroll
            for (int r = 0; r < 16; r++)
                ll[i][j][r] = (int32_t)(((uint32_t)hh[i][j][r] << 16) + ((uint32_t)mid[i][j][r] << 8) +
                                        (uint32_t)ll[i][j][r]);
#pragma unroll
    for (int i = 0; i < RB; i++)
#pragma unroll
        for (int j = 0; j < CB; j++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const v4i v = {ll[i][j][4 * q], ll[i][j][4 * q + 1], ll[i][j][4 * q + 2], ll[i][j][4 * q + 3]};
                __builtin_amdgcn_raw_buffer_store_b128(v, rs, kz * kBlock + wbase + (4 * (CB * i + j) + q) * 1024, 0, 16);
            }
    __builtin_amdgcn_s_waitcnt(0x0070);      // this wave's partial stores complete
    __syncthreads();
    if (threadIdx.x == 0) *ticket = __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (*ticket != nz - 1) return false;
    if (threadIdx.x == 0) __hip_atomic_store(cnt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (uint32_t z = 0; z < nz; z++) {
        if (z == kz) continue;
#pragma unroll
        for (int i = 0; i < RB; i++)
#pragma unroll
            for (int j = 0; j < CB; j++)
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const v4i v = __builtin_amdgcn_raw_buffer_load_b128(rs, z * kBlock + wbase + (4 * (CB * i + j) + q) * 1024, 0, 16);
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        ll[i][j][4 * q + e] = (int32_t)((uint32_t)ll[i][j][4 * q + e] + (uint32_t)v[e]);
                }
    }
#pragma unroll
    for (int i = 0; i < RB; i++)
#pragma unroll
        for (int j = 0; j < CB; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int32_t tot = ll[i][j][r];
                hh[i][j][r] = tot >> 16;
                mid[i][j][r] = (tot >> 8) & 255;
                ll[i][j][r] = tot & 255;
            }
    return true;
}

// ---------------------------------------------------------------- the plane GEMM
// Grid: x = output tiles of one slice (XCD-aware order), y = batch slice, z = k slice (with
// `ksteps` k steps each; 0: no split).  a_slice /
// b_slice: plane bytes per slice (0 = broadcast); the row / column partial sums per SLAB of
// k sit at part[(slice * nslab + s) * lines + line] (slice stride 0 = broadcast).
//
// A workgroup computes a (64 WR) x 128 tile with 2 WR waves in a WR x 2 arrangement, 64 x 64
// outputs each: 2 x 2 blocks of v_mfma_i32_32x32x32_i8 (the i8 MFMA that sustains the full
// rate on gfx950), three int32 accumulators per block (192 registers), so two waves share
// each SIMD:
//   WR = 4, NST = 3: 8 waves, one workgroup per CU, a three-stage LDS ring (144 KiB) with
//     the copies two steps ahead.  Both waves of a SIMD meet at the same barriers, so
//     neither is starved (with two workgroups per CU the older one takes issue priority and
//     the younger finishes alone, at one wave per SIMD);
//   WR = 2, NST = 2: 4 waves, two workgroups per CU, a two-stage ring (64 KiB), for row
//     counts that do not fill 256-row tiles.
// Step k issues the global -> LDS copies (global_load_lds_dwordx4, no registers) of step
// k + NST - 1 at its top, and ends by waiting for this wave's copies of step k + 1 and its
// fragment reads, then for every wave (barrier).  LDS layout: per stage and plane a
// [rows][64 B] tile; row r holds its 16-byte chunk c at chunk c ^ ((r >> 2) & 3), so any
// 16 consecutive rows of one chunk hit 16 distinct bank groups.  A direct copy writes 1 KiB
// (16 rows) per wave instruction, lane l at 16 l.
__device__ __forceinline__ void lds_copy16(const int8_t* g, int8_t* lds_wave_base) {
    __builtin_amdgcn_global_load_lds(g, (__attribute__((address_space(3))) void*)lds_wave_base, 16, 0, 0);
}

// The output tile of workgroup `x` of a slice.  Workgroups are dealt round-robin to the 8 XCDs, each
// with its own L2: the ones of one residue mod 8 take a contiguous run of an order that walks
// strips of `xw` tile columns row by row, so that a run is a block of about xw x xw tiles (xw is
// near the square root of a run's length, gemm_strip) and an XCD reads each operand line once.
// With whole columns as runs (every XCD reading all of A) BERT's 3072-row linears took 29.1 (768 x
// 2304), 15.9 (768 x 768) and 50.2 us (3072 x 768, unsplit); with blocks 28.9, 14.0 and 44.4.
struct TilePos {
    uint32_t id, tr, tc;
};
__device__ __forceinline__ TilePos tile_pos(uint32_t x, uint32_t tiles_r, uint32_t tiles_c, uint32_t xw) {
    const uint32_t ntiles = tiles_r * tiles_c, q = ntiles >> 3, res = x & 7;
    const uint32_t p = res * q + min(res, ntiles & 7) + (x >> 3);
    const uint32_t strip = p / (tiles_r * xw), in = p - strip * tiles_r * xw;
    const uint32_t w = min(xw, tiles_c - strip * xw), row = in / w;
    return TilePos{p, row, strip * xw + in - row * w};
}

template <int WR, int NST, class Epi>
__global__ __launch_bounds__(128 * WR, 8 / (2 * WR)) void gemm_planes_kernel(
    const int8_t* __restrict__ Ahi, const int8_t* __restrict__ Alo, const int32_t* __restrict__ rpart,
    uint64_t a_slice, uint64_t rp_slice, uint32_t a_lines, const int8_t* __restrict__ Bhi,
    const int8_t* __restrict__ Blo, const int32_t* __restrict__ cpart, uint64_t b_slice, uint64_t cp_slice,
    uint32_t b_lines, uint32_t nslab, uint32_t nsum_a, uint32_t tiles_r, uint32_t tiles_c, uint32_t xw, uint32_t kp, int32_t k64,
    uint32_t mode, int32_t* __restrict__ pout, uint32_t ksteps, uint32_t* __restrict__ tcnt, Epi epi) {
    constexpr int TM = 64 * WR;                  // tile rows
    constexpr int NT = 128 * WR;                 // threads
    constexpr int NW = 2 * WR;                   // waves
    constexpr int A_T = TM * BK, B_T = BN * BK;  // plane tile bytes
    constexpr int STAGE = 2 * A_T + 2 * B_T;     // Ah, Al, Bh, Bl
    constexpr int BCP = 8 / NW;                  // 16-row blocks of a B plane per wave
    constexpr int NC = 2 * 2 + 2 * BCP;          // copies per thread and step
    static_assert(NST == 2 || NST == 3, "two or three stages");
    // the stages as separate arrays: with the loop unrolled by NST every access names its
    // stage statically, so the compiler tells the copies in flight into the other stages
    // from the fragment reads
    __shared__ __attribute__((aligned(1024))) int8_t sm0[STAGE];
    __shared__ __attribute__((aligned(1024))) int8_t sm1[STAGE];
    __shared__ __attribute__((aligned(1024))) int8_t sm2[NST == 3 ? STAGE : 16];
    __shared__ int2 rterm[TM], cterm[BN];        // (h, l) halves
    __shared__ uint32_t ticket;                  // kSplitFix: the tile's arrival ticket

    const TilePos tp = tile_pos(blockIdx.x, tiles_r, tiles_c, xw);
    const uint32_t tr = tp.tr, tc = tp.tc;
    const uint32_t bt = blockIdx.y, kz = blockIdx.z;
    const uint32_t kbeg = ksteps ? kz * ksteps : 0;

    const uint32_t t = threadIdx.x, wave = t >> 6, lane = t & 63;
    const uint32_t wr = wave >> 1, wc = wave & 1, l32 = lane & 31, lh = lane >> 5;

    // Row / column terms of the epilogue from the slab partials: the first slab's loads are
    // issued here and used only after the first copies have been issued, so that the two
    // latencies overlap; the other slabs and the LDS writes follow the copies.
    constexpr int TE = (TM + BN + NT - 1) / NT;  // term elements per thread
    int32_t tsum[TE];
#pragma unroll
    for (int q = 0; q < TE; q++) {
        const uint32_t e = t + q * NT;
        tsum[q] = 0;
        if (e < TM + BN)
            tsum[q] = e < TM ? rpart[bt * rp_slice + tr * TM + e] : cpart[bt * cp_slice + tc * BN + (e - TM)];
    }
    auto finish_terms = [&]() {
#pragma unroll
        for (int q = 0; q < TE; q++) {
            const uint32_t e = t + q * NT;
            if (e >= TM + BN) continue;
            const bool is_row = e < TM;
            const uint32_t line = is_row ? tr * TM + e : tc * BN + (e - TM);
            const int32_t* pp = is_row ? rpart + bt * rp_slice + line : cpart + bt * cp_slice + line;
            const uint32_t stride = is_row ? a_lines : b_lines;
            int32_t sum = tsum[q];
            const uint32_t ns = is_row ? nsum_a : nslab;
            for (uint32_t sl = 1; sl < ns; sl++) sum += pp[(uint64_t)sl * stride];
            if (is_row) rterm[e] = make_int2(epi.row_bias(line) - k64 + (sum >> 1), (sum & 1) << 7);
            else cterm[e - TM] = make_int2(sum >> 1, (sum & 1) << 7);
        }
    };

    // copy assignment: wave w fills 16-row blocks 2w, 2w + 1 of each A plane and BCP blocks
    // from BCP w of each B plane; lane l takes row 16 b + l / 4, physical chunk l % 4 =
    // logical chunk (l % 4) ^ swizzle (the swizzle depends on l / 4 only)
    const uint32_t lrow = lane >> 2, cchunk = ((lane & 3) ^ ((lrow >> 2) & 3)) * 16;
    const uint64_t a_base = bt * a_slice + (uint64_t)tr * TM * kp + (uint64_t)kbeg * BK;
    const uint64_t b_base = bt * b_slice + (uint64_t)tc * BN * kp + (uint64_t)kbeg * BK;
    const int8_t* ah_src = Ahi + a_base + (uint64_t)(32 * wave + lrow) * kp + cchunk;
    const int8_t* al_src = Alo + a_base + (uint64_t)(32 * wave + lrow) * kp + cchunk;
    const int8_t* bh_src = Bhi + b_base + (uint64_t)(16 * BCP * wave + lrow) * kp + cchunk;
    const int8_t* bl_src = Blo + b_base + (uint64_t)(16 * BCP * wave + lrow) * kp + cchunk;
    const uint64_t kp16 = (uint64_t)16 * kp;
    const uint32_t a_dst = __builtin_amdgcn_readfirstlane(2048 * wave);
    const uint32_t b_dst = __builtin_amdgcn_readfirstlane(1024 * BCP * wave);

    // fragment read offsets: lane reads row base32 + l32, logical chunk 2 s + lh (substep s)
    const uint32_t sw = (l32 >> 2) & 3;
    const uint32_t fa_row = (wr * 64 + l32) * BK, fb_row = (wc * 64 + l32) * BK;
    const uint32_t ch0 = ((0 + lh) ^ sw) * 16, ch1 = ((2 + lh) ^ sw) * 16;

    v16i hh[2][2], mid[2][2], ll[2][2];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) hh[i][j] = mid[i][j] = ll[i][j] = v16i{};
    v4i ah[2], al[2], bh[2], bl[2];

    const uint32_t nk = ksteps ? min(ksteps, kp / BK - kbeg) : kp / BK;
    // Copy group: the two waves sharing a SIMD (w and w + 4 of 8, as dispatched) issue
    // their copies in different substeps.  With 4 waves per workgroup all are group 0.
    const uint32_t cgrp = NW == 8 ? __builtin_amdgcn_readfirstlane((wave >> 2) & 1) : 0;
    // Copy q of a step (0, 1: A hi; 2, 3: A lo; then B hi, B lo); A rows 16 apart, B blocks.
#define CM_COPY(SM, step, q)                                                                        \
    {                                                                                               \
        const uint64_t k_ = (uint64_t)(step) * BK;                                                  \
        if ((q) < 2) lds_copy16(ah_src + (q) * kp16 + k_, &SM[a_dst + 1024 * (q)]);                 \
        else if ((q) < 4) lds_copy16(al_src + ((q) - 2) * kp16 + k_, &SM[A_T + a_dst + 1024 * ((q) - 2)]); \
        else if ((q) < 4 + BCP)                                                                     \
            lds_copy16(bh_src + ((q) - 4) * kp16 + k_, &SM[2 * A_T + b_dst + 1024 * ((q) - 4)]);    \
        else                                                                                        \
            lds_copy16(bl_src + ((q) - 4 - BCP) * kp16 + k_, &SM[2 * A_T + B_T + b_dst + 1024 * ((q) - 4 - BCP)]); \
    }
    // The copies of slot s (after the s-th group of four MFMAs, 0..7): waves of copy group
    // g issue theirs in slots 4g .. 4g + 3, two, two, then the rest.
#define CM_COPIES(SM, step, slot)                                                 \
    if (!cp_) {                                                                   \
    } else if (((slot) >> 2) == cgrp) {                                           \
        constexpr int s_ = (slot) & 3;                                            \
        if (s_ < 2) { CM_COPY(SM, step, 2 * s_) CM_COPY(SM, step, 2 * s_ + 1) }   \
        else if (NC == 6) { CM_COPY(SM, step, 2 + s_) }                           \
        else { CM_COPY(SM, step, 2 * s_) CM_COPY(SM, step, 2 * s_ + 1) }          \
    }                                                                             \
    __builtin_amdgcn_sched_barrier(0);
#define CM_FRAGS(SM, CH)                                                                   \
    _Pragma("unroll") for (int b = 0; b < 2; b++) {                                        \
        ah[b] = *reinterpret_cast<const v4i*>(&SM[fa_row + b * 32 * BK + CH]);             \
        al[b] = *reinterpret_cast<const v4i*>(&SM[A_T + fa_row + b * 32 * BK + CH]);       \
        bh[b] = *reinterpret_cast<const v4i*>(&SM[2 * A_T + fb_row + b * 32 * BK + CH]);   \
        bl[b] = *reinterpret_cast<const v4i*>(&SM[2 * A_T + B_T + fb_row + b * 32 * BK + CH]); \
    }                                                                                      \
    __builtin_amdgcn_sched_barrier(0);
    // four MFMAs of one limb product over the 2 x 2 blocks
#define CM_MFMA4(ACC, X, Y)                                                                       \
    _Pragma("unroll") for (int i = 0; i < 2; i++) _Pragma("unroll") for (int j = 0; j < 2; j++)   \
        ACC[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(X[i], Y[j], ACC[i][j], 0, 0, 0);       \
    __builtin_amdgcn_sched_barrier(0);
    // One k step on stage SMC while later steps land in the others; SMI receives step
    // kt + NST - 1 when there is one (a wave-uniform branch around each copy).  Two 32-k substeps of 16 MFMAs (hh, mid = h l, ll, mid = l h: no MFMA
    // waits on the one before); the step's copies sit between MFMA groups of the substep
    // of the wave's copy group, so that while one wave of a SIMD spends issue cycles on
    // copies the other has MFMAs to issue, and the sched_barriers keep the compiler from
    // gathering them.  The end of the step waits for this wave's copies of step kt + 1
    // (this step's NC may stay in flight with three stages) and fragment reads, then for
    // every wave.
#define CM_SUBSTEP(SMC, SMI, st, CH, S0)                                          \
    CM_FRAGS(SMC, CH)                                                             \
    CM_MFMA4(hh, ah, bh) CM_COPIES(SMI, st, S0)                                   \
    CM_MFMA4(mid, ah, bl) CM_COPIES(SMI, st, S0 + 1)                              \
    CM_MFMA4(ll, al, bl) CM_COPIES(SMI, st, S0 + 2)                               \
    CM_MFMA4(mid, al, bh) CM_COPIES(SMI, st, S0 + 3)
#define CM_STEP(kt, SMC, SMI)                                                     \
    {                                                                             \
        const uint32_t st_ = (kt) + NST - 1;                                      \
        const bool cp_ = st_ < nk;                                                \
        CM_SUBSTEP(SMC, SMI, st_, ch0, 0)                                         \
        CM_SUBSTEP(SMC, SMI, st_, ch1, 4)                                         \
        if (NST == 3 && cp_) __builtin_amdgcn_s_waitcnt(0x0070 | NC);             \
        else __builtin_amdgcn_s_waitcnt(0x0070);                                  \
        __builtin_amdgcn_s_barrier();                                             \
    }
#define CM_ISSUE(SM, step)                                                        \
    _Pragma("unroll") for (int q_ = 0; q_ < NC; q_++) CM_COPY(SM, step, q_)

    uint32_t kt = 0;
    if constexpr (NST == 3) {
        CM_ISSUE(sm0, 0)
        if (nk > 1) {
            CM_ISSUE(sm1, 1)
            finish_terms();
            __builtin_amdgcn_s_waitcnt(0x0070 | NC);
        } else {
            finish_terms();
            __builtin_amdgcn_s_waitcnt(0x0070);
        }
        __builtin_amdgcn_s_barrier();
        for (; kt + 3 <= nk; kt += 3) {
            CM_STEP(kt, sm0, sm2)
            CM_STEP(kt + 1, sm1, sm0)
            CM_STEP(kt + 2, sm2, sm1)
        }
        if (kt < nk) CM_STEP(kt, sm0, sm2)
        if (kt + 1 < nk) CM_STEP(kt + 1, sm1, sm0)
    } else {
        CM_ISSUE(sm0, 0)
        finish_terms();
        __builtin_amdgcn_s_waitcnt(0x0070);
        __builtin_amdgcn_s_barrier();
        for (; kt + 2 <= nk; kt += 2) {
            CM_STEP(kt, sm0, sm1)
            CM_STEP(kt + 1, sm1, sm0)
        }
        if (kt < nk) CM_STEP(kt, sm0, sm1)
    }
    __builtin_amdgcn_s_waitcnt(0x0070);      // no copy may land after the workgroup ends
#undef CM_ISSUE
#undef CM_STEP
#undef CM_SUBSTEP
#undef CM_MFMA4
#undef CM_FRAGS
#undef CM_COPIES
#undef CM_COPY

    // ---- epilogue: one uniform dispatch to the store routine of this mode
    const uint32_t row0 = tr * TM, col0 = tc * BN;
    if (mode == kSplitFix) {
        // the slices' partials meet in the last slice to arrive; the others are done
        const uint64_t tile_id = (uint64_t)bt * tiles_r * tiles_c + tp.id;
        if (!split_fixup<NW, 2, 2>(hh, mid, ll, pout + tile_id * gridDim.z * (TM * BN), gridDim.z, kz, wave, lane,
                             tcnt + tile_id, &ticket))
            return;
        mode = kWrap;
    }
#define CM_STORE(M, P) store_wave_tile<M, P, 2, 2>(hh, mid, ll, rterm, cterm, bt, row0, col0, wr, wc, l32, lh, epi)
    const TileBase tb = epi.tile_base(bt, row0, col0, TM, BN);
    if (tb.base != nullptr) {           // a whole tile: the lean store
        if (mode == kWrap) store_wave_fast<kWrap, 2, 2>(hh, mid, ll, rterm, cterm, tb.base, tb.ld, wr, wc, l32, lh, epi.lo, epi.hi);
        else if (mode == kSatNarrow)
            store_wave_fast<kSatNarrow, 2, 2>(hh, mid, ll, rterm, cterm, tb.base, tb.ld, wr, wc, l32, lh, epi.lo, epi.hi);
        else store_wave_fast<kSatWide, 2, 2>(hh, mid, ll, rterm, cterm, tb.base, tb.ld, wr, wc, l32, lh, epi.lo, epi.hi);
    } else if (mode == kSatNarrow) {
        if (epi.pairs) CM_STORE(kSatNarrow, true); else CM_STORE(kSatNarrow, false);
    } else if (mode == kWrap) {
        if (epi.pairs) CM_STORE(kWrap, true); else CM_STORE(kWrap, false);
    } else {
        if (epi.pairs) CM_STORE(kSatWide, true); else CM_STORE(kSatWide, false);
    }
#undef CM_STORE
}

// ---------------------------------------------------------------- the plane GEMM, few tiles
// The same product for outputs of few tiles (a 128-token layer, a prompt's projections, a
// network's 7 x 7 and 14 x 14 planes), where the kernel above is bound by latency: its two-stage
// ring gives a copy less than one k step to arrive, a wavefront's fragment reads stall its own
// MFMAs, and its 128 x 128 tiles leave most compute units idle.  Here a workgroup of WR x WC
// waves computes (32 RB WR) x (32 CB WC) outputs over a ring of NST = 4 stages:
//   - copies run NST - 1 steps ahead, so that with few steps nearly all of k is in flight at once;
//   - a wavefront reads the next step's fragments (both 32-k substeps) while its MFMAs of this step
//     run, from a stage that landed one step earlier: one barrier a step, and no MFMA waits on LDS.
// Stage, plane and swizzle layout as above; the 1 KiB copies of a stage (16 rows each: A hi, A lo,
// B hi, B lo) are dealt to the waves in equal runs, each from its own uniform base address.
template <int N>
__device__ __forceinline__ void wait_copies() {            // at most N of this wave's copies outstanding, LDS reads done
    static_assert(N >= 0 && N < 64, "vmcnt is six bits");
    __builtin_amdgcn_s_waitcnt(0x0070 | (N & 15) | ((N >> 4) << 14));
}

// The copies (NC a step) of all but the newest `later` (at most MAX) steps have landed.
template <int NC, int MAX>
__device__ __forceinline__ void wait_steps(uint32_t later) {
    if constexpr (MAX == 0) wait_copies<0>();
    else if (later >= MAX) wait_copies<MAX * NC>();
    else wait_steps<NC, MAX - 1>(later);
}

template <int RB, int CB, int WR, int WC, class Epi>
__global__ __launch_bounds__(64 * WR * WC, 2) void gemm_ring_kernel(
    const int8_t* __restrict__ Ahi, const int8_t* __restrict__ Alo, const int32_t* __restrict__ rpart,
    uint64_t a_slice, uint64_t rp_slice, uint32_t a_lines, const int8_t* __restrict__ Bhi,
    const int8_t* __restrict__ Blo, const int32_t* __restrict__ cpart, uint64_t b_slice, uint64_t cp_slice,
    uint32_t b_lines, uint32_t nslab, uint32_t nsum_a, uint32_t tiles_r, uint32_t tiles_c, uint32_t xw, uint32_t kp, int32_t k64,
    uint32_t mode, int32_t* __restrict__ pout, uint32_t ksteps, uint32_t* __restrict__ tcnt, Epi epi) {
    constexpr int TM = 32 * RB * WR, TN = 32 * CB * WC;
    constexpr int NST = 4;                             // stages (even: the fragment registers alternate)
    constexpr int NW = WR * WC, NT = 64 * NW;
    constexpr int A_T = TM * BK, B_T = TN * BK;        // plane tile bytes
    constexpr int STAGE = 2 * A_T + 2 * B_T;           // Ah, Al, Bh, Bl
    constexpr int NC = STAGE / 1024 / NW;              // copies per wave and step
    static_assert(STAGE % (1024 * NW) == 0, "equal copies per wave");
    static_assert(NC * (NST - 1) < 64, "vmcnt is six bits");
    // separate arrays: the compiler then tells the copies in flight from the fragment reads
    __shared__ __attribute__((aligned(1024))) int8_t sm0[STAGE], sm1[STAGE], sm2[STAGE], sm3[STAGE];
    __shared__ int2 rterm[TM], cterm[TN];              // (h, l) halves
    __shared__ uint32_t ticket;                        // kSplitFix: the tile's arrival ticket

    const TilePos tp = tile_pos(blockIdx.x, tiles_r, tiles_c, xw);
    const uint32_t tr = tp.tr, tc = tp.tc;
    const uint32_t bt = blockIdx.y, kz = blockIdx.z;
    const uint32_t kbeg = ksteps ? kz * ksteps : 0;
    const uint32_t nk = ksteps ? min(ksteps, kp / BK - kbeg) : kp / BK;

    const uint32_t t = threadIdx.x, lane = t & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const uint32_t wr = wave / WC, wc = wave % WC, l32 = lane & 31, lh = lane >> 5;

    // copies: wave w takes the 16-row blocks NC w .. NC w + NC - 1 of a stage; lane l row l / 4,
    // physical chunk l % 4 = logical chunk (l % 4) ^ swizzle
    const uint32_t lrow = lane >> 2, cchunk = ((lane & 3) ^ ((lrow >> 2) & 3)) * 16;
    const uint32_t voff = lrow * kp + cchunk;
    const uint64_t a_base = bt * a_slice + (uint64_t)tr * TM * kp + (uint64_t)kbeg * BK;
    const uint64_t b_base = bt * b_slice + (uint64_t)tc * TN * kp + (uint64_t)kbeg * BK;
    const int8_t* src[NC];
#pragma unroll
    for (int q = 0; q < NC; q++) {
        uint32_t blk = NC * wave + q;
        if (blk < 2 * TM / 16) {
            const bool low = blk >= TM / 16;
            blk -= low ? TM / 16 : 0;
            src[q] = (low ? Alo : Ahi) + a_base + (uint64_t)blk * 16 * kp;
        } else {
            blk -= 2 * TM / 16;
            const bool low = blk >= TN / 16;
            blk -= low ? TN / 16 : 0;
            src[q] = (low ? Blo : Bhi) + b_base + (uint64_t)blk * 16 * kp;
        }
    }
    auto issue = [&](int8_t* sm, uint32_t step) {
#pragma unroll
        for (int q = 0; q < NC; q++) lds_copy16(src[q] + (uint64_t)step * BK + voff, sm + (NC * wave + q) * 1024);
    };
    // the partial line sums: the first twelve of a line are loaded before the copies go out and used
    // after them (a load issued behind the copies would be waited for behind them)
    constexpr int TE = (TM + TN + NT - 1) / NT, TP = 12;
    int32_t tpart[TE][TP];
    auto term_src = [&](uint32_t e, uint32_t& stride, uint32_t& ns) -> const int32_t* {
        const bool is_row = e < TM;
        stride = is_row ? a_lines : b_lines;
        ns = is_row ? nsum_a : nslab;
        return is_row ? rpart + bt * rp_slice + tr * TM + e : cpart + bt * cp_slice + tc * TN + (e - TM);
    };
#pragma unroll
    for (int q = 0; q < TE; q++) {
        const uint32_t e = t + q * NT;
        if (e >= TM + TN) continue;
        uint32_t stride, ns;
        const int32_t* pp = term_src(e, stride, ns);
#pragma unroll
        for (int i = 0; i < 4; i++) tpart[q][i] = pp[(uint64_t)min((uint32_t)i, ns - 1) * stride];
        if (ns > 4) {
#pragma unroll
            for (int i = 4; i < TP; i++) tpart[q][i] = pp[(uint64_t)min((uint32_t)i, ns - 1) * stride];
        }
    }
#define CM_ST(i) ((i) % NST == 0 ? sm0 : (i) % NST == 1 ? sm1 : (i) % NST == 2 ? sm2 : sm3)
    issue(sm0, 0);
    if (1 < nk) issue(sm1, 1);
    if (2 < nk) issue(sm2, 2);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < TE; q++) {
        const uint32_t e = t + q * NT;
        if (e >= TM + TN) continue;
        uint32_t stride, ns;
        const int32_t* pp = term_src(e, stride, ns);
        int32_t sum = 0;
#pragma unroll
        for (int i = 0; i < 4; i++) sum += (uint32_t)i < ns ? tpart[q][i] : 0;
        if (ns > 4) {
#pragma unroll
            for (int i = 4; i < TP; i++) sum += (uint32_t)i < ns ? tpart[q][i] : 0;
            for (uint32_t sl = TP; sl < ns; sl++) sum += pp[(uint64_t)sl * stride];
        }
        if (e < TM) rterm[e] = make_int2(epi.row_bias(tr * TM + e) - k64 + (sum >> 1), (sum & 1) << 7);
        else cterm[e - TM] = make_int2(sum >> 1, (sum & 1) << 7);
    }

    const uint32_t sw = (l32 >> 2) & 3;
    const uint32_t fa_row = (wr * (32 * RB) + l32) * BK, fb_row = (wc * (32 * CB) + l32) * BK;
    const uint32_t ch[2] = {((0 + lh) ^ sw) * 16, ((2 + lh) ^ sw) * 16};
    struct Frags { v4i ah[2][RB], al[2][RB], bh[2][CB], bl[2][CB]; };
    auto read = [&](const int8_t* sm, Frags& f) {
#pragma unroll
        for (int s = 0; s < 2; s++) {
#pragma unroll
            for (int b = 0; b < RB; b++) {
                f.ah[s][b] = *reinterpret_cast<const v4i*>(sm + fa_row + b * 32 * BK + ch[s]);
                f.al[s][b] = *reinterpret_cast<const v4i*>(sm + A_T + fa_row + b * 32 * BK + ch[s]);
            }
#pragma unroll
            for (int b = 0; b < CB; b++) {
                f.bh[s][b] = *reinterpret_cast<const v4i*>(sm + 2 * A_T + fb_row + b * 32 * BK + ch[s]);
                f.bl[s][b] = *reinterpret_cast<const v4i*>(sm + 2 * A_T + B_T + fb_row + b * 32 * BK + ch[s]);
            }
        }
    };
    v16i hh[RB][CB], mid[RB][CB], ll[RB][CB];
#pragma unroll
    for (int i = 0; i < RB; i++)
#pragma unroll
        for (int j = 0; j < CB; j++) hh[i][j] = mid[i][j] = ll[i][j] = v16i{};
    auto mfma = [&](const Frags& f) {
#pragma unroll
        for (int s = 0; s < 2; s++) {
#define CM_MFMAS(ACC, X, Y)                                                       \
    _Pragma("unroll") for (int i = 0; i < RB; i++) _Pragma("unroll") for (int j = 0; j < CB; j++) \
        ACC[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(f.X[s][i], f.Y[s][j], ACC[i][j], 0, 0, 0);
            CM_MFMAS(hh, ah, bh)
            CM_MFMAS(mid, ah, bl)
            CM_MFMAS(ll, al, bl)
            CM_MFMAS(mid, al, bh)
#undef CM_MFMAS
        }
    };
    // Every wave waits for its copies of step kt + 1 (those of up to NST - 3 later steps stay in
    // flight) and its fragment reads of step kt, then for the other waves: stage kt + 1 is
    // whole, and stage kt - 1, whose fragments every wave has consumed, takes step kt + NST - 1.
    auto meet = [&](uint32_t kt) {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        wait_steps<NC, NST - 3>(nk - 2 - kt);          // kt + 1 < nk
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" ::: "memory");
    };
    Frags f0, f1;
    {   // stage 0: the copies of at most NST - 2 later steps stay in flight
        __builtin_amdgcn_sched_barrier(0);
        wait_steps<NC, NST - 2>(nk - 1);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" ::: "memory");
    }
    read(sm0, f0);
    // (the wait for CUR stands outside the branch, where the compiler sees it on every path)
#define CM_RSTEP(I, CUR, NXT)                                                     \
    __builtin_amdgcn_s_waitcnt(0xC07F);                                           \
    if (kt + 1 < nk) {                                                            \
        meet(kt);                                                                 \
        if (kt + NST - 1 < nk) issue(CM_ST((I) + NST - 1), kt + NST - 1);         \
        read(CM_ST((I) + 1), NXT);                                                \
    }                                                                             \
    mfma(CUR);                                                                    \
    if (++kt >= nk) break;
    for (uint32_t kt = 0;;) {
        CM_RSTEP(0, f0, f1)
        CM_RSTEP(1, f1, f0)
        CM_RSTEP(2, f0, f1)
        CM_RSTEP(3, f1, f0)
    }
#undef CM_RSTEP
#undef CM_ST

    // ---- epilogue (every copy has landed: the last step waited for it)
    const uint32_t row0 = tr * TM, col0 = tc * TN;
    if (mode == kSplitFix) {
        const uint64_t tile_id = (uint64_t)bt * tiles_r * tiles_c + tp.id;
        if (!split_fixup<NW, RB, CB>(hh, mid, ll, pout + tile_id * gridDim.z * (TM * TN), gridDim.z, kz, wave, lane,
                                     tcnt + tile_id, &ticket))
            return;
        mode = kWrap;
    }
#define CM_STORE(M, P) store_wave_tile<M, P, RB, CB>(hh, mid, ll, rterm, cterm, bt, row0, col0, wr, wc, l32, lh, epi)
#define CM_STORE_FAST(M) \
    store_wave_fast<M, RB, CB>(hh, mid, ll, rterm, cterm, tb.base, tb.ld, wr, wc, l32, lh, epi.lo, epi.hi)
    const TileBase tb = epi.tile_base(bt, row0, col0, TM, TN);
    if (tb.base != nullptr) {
        if (mode == kWrap) CM_STORE_FAST(kWrap);
        else if (mode == kSatNarrow) CM_STORE_FAST(kSatNarrow);
        else CM_STORE_FAST(kSatWide);
    } else if (mode == kSatNarrow) {
        if (epi.pairs) CM_STORE(kSatNarrow, true); else CM_STORE(kSatNarrow, false);
    } else if (mode == kWrap) {
        if (epi.pairs) CM_STORE(kWrap, true); else CM_STORE(kWrap, false);
    } else {
        if (epi.pairs) CM_STORE(kSatWide, true); else CM_STORE(kSatWide, false);
    }
#undef CM_STORE_FAST
#undef CM_STORE
}

// ---------------------------------------------------------------- 1x1 convolutions, pixels in registers
// A 1x1 stride-1 convolution is the product of the weights' planes and each image's [channels][pixels]
// matrix.  Folding the images into byte planes first (split_fold*) writes and reads the whole input
// again and costs a launch; here a wave of 32 output channels x 32 PX pixels reads its pixels straight
// into the MFMA operand's layout: a lane's operand is 16 channels of one pixel, so it loads its PX
// pixels in 16 channels (32 lanes side by side), transposes them with byte permutes and adds the
// pixel's byte sums (v_dot4).  The weights' operand is 16 bytes of each plane.  Nothing is staged and
// no barrier stands in the loop; D steps of 32 channels are in flight (a step's rows lie a plane
// apart in HBM).  KW waves share one output tile's channels where the tiles alone leave the chip idle:
// they exchange their accumulators through LDS and each stores 16 / KW of a lane's rows.  The launch
// bounds keep a wave within 256 registers, so that the accumulators stay where the epilogue's vector
// instructions read them (in AGPRs, 3 moves an element: 16 -> 96 at 32 x 112 x 112 37 us, 28 without).
// Measured at batch 32, us, against a workgroup that split its 64 x 64 tile's pixels through LDS: 96 ->
// 24 at 56 x 56 7.9 (15.9; its 24 MB 4.0 at 6 TB/s), 576 -> 96 at 14 x 14 9.7 (11.8), 960 -> 320 at 7 x 7
// 11.4 (16.6), 512 -> 512 at 28 x 28 55.8 (65.5).
// A wave's pixels of 16 channels from c0 on, PX a lane: one 32-bit offset a lane (the lane's pixel and
// channel; below 2^32 bytes, the dispatch's rule) on scalar row addresses.  Channels at and past K read
// some channel below it (their weights' planes are 0 there).
template <int PX, bool RAG>
struct PointPx {
    typedef typename std::conditional<PX == 1, uint16_t, uint32_t>::type Px;
    Px b[16];
    __device__ __forceinline__ void load(const int16_t* x, uint32_t pix, uint32_t row, uint32_t c0, uint32_t K) {
        const uint32_t off = pix + (RAG ? 0u : min(c0, K - 16) * row);
#pragma unroll
        for (uint32_t r = 0; r < 16; r++) {
            const char* xr = reinterpret_cast<const char*>(x) + (RAG ? 0u : (uint64_t)(r * row));
            __builtin_memcpy(&b[r], xr + (RAG ? off + min(c0 + r, K - 1) * row : off), sizeof(Px));
        }
    }
    // the byte planes of pixel j in channels c0 + 4 g .. + 3 (plane bytes as the splits write them), and
    // their sums over the channels below K
    __device__ __forceinline__ void planes(v4i (&bh)[PX], v4i (&bl)[PX], int32_t (&sh)[PX], int32_t (&sl)[PX],
                                           uint32_t c0, uint32_t K) const {
#pragma unroll
        for (int g = 0; g < 4; g++) {
            uint32_t one = 0x01010101u;
            if constexpr (RAG) one = c0 + 4 * g >= K ? 0u : one >> (8 * (4 - min(K - c0 - 4 * g, 4u)));
            else one = c0 >= K ? 0u : one;
            if constexpr (PX == 1) {
                const uint32_t a = (uint32_t)b[4 * g] | (uint32_t)b[4 * g + 1] << 16,
                               c = (uint32_t)b[4 * g + 2] | (uint32_t)b[4 * g + 3] << 16;
                bh[0][g] = (int)__builtin_amdgcn_perm(c, a, 0x07050301u);
                bl[0][g] = (int)(__builtin_amdgcn_perm(c, a, 0x06040200u) ^ 0x80808080u);
            } else {
                const uint32_t xh = __builtin_amdgcn_perm(b[4 * g + 1], b[4 * g], 0x07030501u),
                               yh = __builtin_amdgcn_perm(b[4 * g + 3], b[4 * g + 2], 0x07030501u),
                               xl = __builtin_amdgcn_perm(b[4 * g + 1], b[4 * g], 0x06020400u),
                               yl = __builtin_amdgcn_perm(b[4 * g + 3], b[4 * g + 2], 0x06020400u);
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    const uint32_t sel = j ? 0x07060302u : 0x05040100u;
                    bh[j][g] = (int)__builtin_amdgcn_perm(yh, xh, sel);
                    bl[j][g] = (int)(__builtin_amdgcn_perm(yl, xl, sel) ^ 0x80808080u);
                }
            }
#pragma unroll
            for (int j = 0; j < PX; j++) {
                sh[j] = __builtin_amdgcn_sdot4(bh[j][g], (int)one, sh[j], false);
                sl[j] = __builtin_amdgcn_sdot4(bl[j][g], (int)one, sl[j], false);
            }
        }
    }
};

// The results of a lane's PX pixels in one row: rows of terms (rh, rl), columns (ch, cl), as recombine; two
// pixels are saturated, packed and clamped in pairs.  kSatTiny: K <= 256, where 2^8 HH needs no clamp.
constexpr uint32_t kSatTiny = 4;
typedef short v2s __attribute__((ext_vector_type(2)));
template <uint32_t MODE, int PX>
__device__ __forceinline__ void point_out(int16_t* dst, const int32_t (&hh)[PX], const int32_t (&mid)[PX], const int32_t (&ll)[PX],
                                          int2 rt, const int32_t (&ch)[PX], const int32_t (&cl)[PX], int32_t lo, int32_t hi) {
    int32_t q[PX];
#pragma unroll
    for (int j = 0; j < PX; j++) {
        if constexpr (MODE == kSatTiny) q[j] = (int32_t)((uint32_t)hh[j] << 8) + (mid[j] + rt.x + ch[j]) + ((ll[j] + rt.y + cl[j]) >> 8);
        else q[j] = recombine<MODE>(hh[j], mid[j], ll[j], rt.x + ch[j], rt.y + cl[j], -32768, 32767);
    }
    if constexpr (PX == 1) {
        *dst = (int16_t)clamp_i32(q[0], lo, hi);
    } else {
        v2s o = __builtin_amdgcn_cvt_pk_i16(q[0], q[1]);
        o = __builtin_elementwise_min(__builtin_elementwise_max(o, v2s{(short)lo, (short)lo}), v2s{(short)hi, (short)hi});
        __builtin_memcpy(dst, &o, 4);
    }
}

template <int PX, int KW, bool RAG>
__global__ __launch_bounds__(64 * KW, PX == 2 ? 2 : 3) void conv_point_kernel(
    const int8_t* __restrict__ Ahi, const int8_t* __restrict__ Alo, const int32_t* __restrict__ rpart,
    uint32_t a_lines, uint32_t nsum_a, const int16_t* __restrict__ x, uint32_t K, uint32_t plane, uint32_t cols,
    uint32_t tiles_r, uint32_t tiles_c, uint32_t kp, uint32_t mode, EpiConv epi) {
    constexpr int RW = 16 / KW, D = PX == 1 ? 3 : 2;
    const uint32_t kpart = KW == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t lane = threadIdx.x & 63, l32 = lane & 31, lh = lane >> 5;
    // the row tiles of one pixel tile run on one XCD, one after the other (its L2 holds the pixels)
    const TilePos tp = tile_pos(blockIdx.x, tiles_r, tiles_c, 1);
    const uint32_t tr = tp.tr;
    const uint32_t col = (tp.tc * 32 + l32) * PX;                            // pixels over all images
    const bool live = col < cols;
    const uint32_t c = min(col, cols - PX), img = c / plane, p = c - img * plane;
    const uint32_t nk = (K + 31) / 32, k0 = nk * kpart / KW, k1 = nk * (kpart + 1) / KW;   // this wave's steps
    const uint32_t pix = 2 * (img * K * plane + p), row = 2 * plane;
    const int8_t* const ah = Ahi + (uint64_t)(tr * 32 + l32) * kp + 16 * lh;
    const int8_t* const al = Alo + (uint64_t)(tr * 32 + l32) * kp + 16 * lh;
    struct Step { v4i ah, al; PointPx<PX, RAG> x; };
    auto load = [&](Step& v, uint32_t k) {
        v.ah = *reinterpret_cast<const v4i*>(ah + k * 32);
        v.al = *reinterpret_cast<const v4i*>(al + k * 32);
        v.x.load(x, pix, row, 32 * k + 16 * lh, K);
    };
    v16i hh[PX], mid[PX], ll[PX];
    int32_t sh[PX], sl[PX];
#pragma unroll
    for (int j = 0; j < PX; j++) {
        hh[j] = mid[j] = ll[j] = v16i{};
        sh[j] = sl[j] = 0;
    }
    auto step = [&](const Step& v, uint32_t k) {
        v4i bh[PX], bl[PX];
        v.x.planes(bh, bl, sh, sl, 32 * k + 16 * lh, K);
#pragma unroll
        for (int j = 0; j < PX; j++) {
            hh[j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(v.ah, bh[j], hh[j], 0, 0, 0);
            mid[j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(v.ah, bl[j], mid[j], 0, 0, 0);
            ll[j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(v.al, bl[j], ll[j], 0, 0, 0);
        }
#pragma unroll
        for (int j = 0; j < PX; j++) mid[j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(v.al, bh[j], mid[j], 0, 0, 0);
    };
    Step v[D];
#pragma unroll
    for (int i = 0; i < D; i++)
        if (k0 + i < k1) load(v[i], k0 + i);
    int32_t rsum = 0;                                                        // the lane's row's terms
    for (uint32_t s = 0; s < nsum_a; s++) rsum += rpart[(uint64_t)s * a_lines + tr * 32 + l32];
    const int32_t rb = epi.row_bias(tr * 32 + l32);
    for (uint32_t k = k0; k < k1;) {
#pragma unroll
        for (int i = 0; i < D; i++) {
            step(v[i], k);
            if (k + D < k1) load(v[i], k + D);
            if (++k >= k1) break;
        }
    }

    // terms of the columns and the rows: x = 256 h + l + 128 (recombine)
    __shared__ int2 rterm[32];
    __shared__ int32_t xch[KW > 1 ? KW * PX * 49 * 64 : 1];                  // [wave][pixel][3 accumulators x 16, sum][lane]
    if (kpart == 0 && lh == 0) rterm[l32] = make_int2(rb - (int32_t)(64 * K) + (rsum >> 1), (rsum & 1) << 7);
    int32_t cs[PX];
#pragma unroll
    for (int j = 0; j < PX; j++) {
        cs[j] = (sh[j] << 8) + sl[j];
        cs[j] += __shfl_xor(cs[j], 32, 64);
    }
    if constexpr (KW > 1) {
        // wave kpart keeps rows RW kpart .. of every lane and hands the others theirs
#pragma unroll
        for (int j = 0; j < PX; j++) {
#pragma unroll
            for (int r = 0; r < 16; r++) {
                xch[((kpart * PX + j) * 49 + 3 * r) * 64 + lane] = hh[j][r];
                xch[((kpart * PX + j) * 49 + 3 * r + 1) * 64 + lane] = mid[j][r];
                xch[((kpart * PX + j) * 49 + 3 * r + 2) * 64 + lane] = ll[j][r];
            }
            xch[((kpart * PX + j) * 49 + 48) * 64 + lane] = cs[j];
        }
        __syncthreads();
    } else {
        __builtin_amdgcn_wave_barrier();
    }
    int32_t ch[PX], cl[PX];
    int32_t fh[RW][PX], fm[RW][PX], fl[RW][PX];
#pragma unroll
    for (int j = 0; j < PX; j++) {
        int32_t s = cs[j];
        if constexpr (KW > 1) {
            s = 0;
#pragma unroll
            for (int w = 0; w < KW; w++) s += xch[((w * PX + j) * 49 + 48) * 64 + lane];
        }
        s += (int32_t)(128 * K);
        ch[j] = s >> 1;
        cl[j] = (s & 1) << 7;
#pragma unroll
        for (int r = 0; r < RW; r++) {
            if constexpr (KW == 1) {
                fh[r][j] = hh[j][r];
                fm[r][j] = mid[j][r];
                fl[r][j] = ll[j][r];
            } else {
                const uint32_t q = kpart * RW + r;
                fh[r][j] = fm[r][j] = fl[r][j] = 0;
#pragma unroll
                for (int w = 0; w < KW; w++) {
                    fh[r][j] += xch[((w * PX + j) * 49 + 3 * q) * 64 + lane];
                    fm[r][j] += xch[((w * PX + j) * 49 + 3 * q + 1) * 64 + lane];
                    fl[r][j] += xch[((w * PX + j) * 49 + 3 * q + 2) * 64 + lane];
                }
            }
        }
    }
    if (!live) return;                                                       // no barrier follows
    const bool flat = epi.cn == 0 && tr * 32 + 32 <= epi.rows;               // uniform: rows cs apart, all inside
    int16_t* const yl = epi.y + img * epi.img + (uint64_t)(tr * 32 + 4 * lh) * epi.cs + p;
    auto store = [&](auto m) {
        constexpr uint32_t MODE = decltype(m)::value;
#pragma unroll
        for (int r = 0; r < RW; r++) {
            const uint32_t q = kpart * RW + r, rl = 8 * (q / 4) + q % 4;
            int16_t* dst = yl + (uint64_t)rl * epi.cs;
            if (!flat) {
                dst = epi.row_ptr(img, tr * 32 + 4 * lh + rl);
                if (dst == nullptr) continue;
                dst += p;
            }
            point_out<MODE, PX>(dst, fh[r], fm[r], fl[r], rterm[4 * lh + rl], ch, cl, epi.lo, epi.hi);
        }
    };
    if (mode == kWrap) store(std::integral_constant<uint32_t, kWrap>{});
    else if (mode == kSatNarrow) store(std::integral_constant<uint32_t, kSatNarrow>{});
    else if (mode == kSatTiny) store(std::integral_constant<uint32_t, kSatTiny>{});
    else store(std::integral_constant<uint32_t, kSatWide>{});
}

constexpr uint32_t kPointTiles = 3;              // row tiles of a wave, at most

// The same product of at most 32 NK channels (a network's expansions, whose outputs outweigh everything
// else): a wave keeps its 32 pixels' operands in registers and takes gt row tiles one after the
// other, the next tile's weights in flight, so that the pixels' latency and transposition are paid
// once for all of them.
template <int NK, bool RAG>
__global__ __launch_bounds__(256, NK > 1 ? 3 : 4) void conv_point_wide_kernel(
    const int8_t* __restrict__ Ahi, const int8_t* __restrict__ Alo, const int32_t* __restrict__ rpart,
    const int16_t* __restrict__ x, uint32_t K, uint32_t plane, uint32_t cols, uint32_t blocks_r, uint32_t blocks_c,
    uint32_t tiles_r, uint32_t gt, uint32_t kp, uint32_t mode, EpiConv epi) {
    __shared__ int2 rterm[kPointTiles * 32];
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l32 = lane & 31, lh = lane >> 5;
    const TilePos tp = tile_pos(blockIdx.x, blocks_r, blocks_c, 1);
    const uint32_t t0 = tp.tr * gt, t1 = min(t0 + gt, tiles_r);
    const uint32_t col = (tp.tc * 4 + wave) * 32 + l32;      // a pixel a lane, over all images (two measured the same)
    const bool live = col < cols;
    const uint32_t c = min(col, cols - 1), img = c / plane, p = c - img * plane;
    const uint32_t pix = 2 * (img * K * plane + p), row = 2 * plane;
    const uint64_t aoff = (uint64_t)(t0 * 32 + l32) * kp + 16 * lh;
    PointPx<1, RAG> px[NK];
#pragma unroll
    for (int k = 0; k < NK; k++) px[k].load(x, pix, row, 32 * k + 16 * lh, K);
    v4i ah[NK], al[NK];
    auto load_a = [&](uint32_t t) {
#pragma unroll
        for (int k = 0; k < NK; k++) {
            ah[k] = *reinterpret_cast<const v4i*>(Ahi + aoff + (uint64_t)(t - t0) * 32 * kp + 32 * k);
            al[k] = *reinterpret_cast<const v4i*>(Alo + aoff + (uint64_t)(t - t0) * 32 * kp + 32 * k);
        }
    };
    load_a(t0);
    if (const uint32_t i = threadIdx.x; i < (t1 - t0) * 32) {
        const int32_t sum = rpart[t0 * 32 + i];                              // one slab: K <= 1024
        rterm[i] = make_int2(epi.row_bias(t0 * 32 + i) - (int32_t)(64 * K) + (sum >> 1), (sum & 1) << 7);
    }
    __syncthreads();
    v4i bh[NK][1], bl[NK][1];
    int32_t sh[1] = {0}, sl[1] = {0};
#pragma unroll
    for (int k = 0; k < NK; k++) px[k].planes(bh[k], bl[k], sh, sl, 32 * k + 16 * lh, K);
    int32_t s = (sh[0] << 8) + sl[0];
    s += __shfl_xor(s, 32, 64);
    s += (int32_t)(128 * K);                                                 // x = 256 h + l + 128
    const int32_t ch[1] = {s >> 1}, cl[1] = {(s & 1) << 7};
    int16_t* const yb = epi.y + img * epi.img + (uint64_t)(4 * lh) * epi.cs + p;
    auto tiles = [&](auto m) {
        constexpr uint32_t MODE = decltype(m)::value;
        for (uint32_t t = t0; t < t1; t++) {
            v16i hh = v16i{}, mid = v16i{}, ll = v16i{};
#pragma unroll
            for (int k = 0; k < NK; k++) {
                hh = __builtin_amdgcn_mfma_i32_32x32x32_i8(ah[k], bh[k][0], hh, 0, 0, 0);
                mid = __builtin_amdgcn_mfma_i32_32x32x32_i8(ah[k], bl[k][0], mid, 0, 0, 0);
                ll = __builtin_amdgcn_mfma_i32_32x32x32_i8(al[k], bl[k][0], ll, 0, 0, 0);
                mid = __builtin_amdgcn_mfma_i32_32x32x32_i8(al[k], bh[k][0], mid, 0, 0, 0);
            }
            if (t + 1 < t1) load_a(t + 1);
            if (live) {
                const bool flat = epi.cn == 0 && t * 32 + 32 <= epi.rows;    // uniform: rows cs apart, all inside
                int16_t* const yl = yb + (uint64_t)t * 32 * epi.cs;
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const uint32_t rl = 8 * (r / 4) + r % 4;
                    int16_t* dst = yl + (uint64_t)rl * epi.cs;
                    if (!flat) {
                        dst = epi.row_ptr(img, t * 32 + 4 * lh + rl);
                        if (dst == nullptr) continue;
                        dst += p;
                    }
                    const int32_t h[1] = {hh[r]}, m2[1] = {mid[r]}, l[1] = {ll[r]};
                    point_out<MODE, 1>(dst, h, m2, l, rterm[(t - t0) * 32 + 4 * lh + rl], ch, cl, epi.lo, epi.hi);
                }
            }
        }
    };
    if (mode == kWrap) tiles(std::integral_constant<uint32_t, kWrap>{});
    else tiles(std::integral_constant<uint32_t, kSatTiny>{});
}

// ---------------------------------------------------------------- standard conv, few taps
// A standard convolution whose taps per output (in_ch kh kw <= 80) are few -- a network's stem
// over its 1 .. 4 input channels, the 1x1 convolutions of up to 80 channels whose weights come packed
// with the call (split once, they run from their pixels, above) -- straight on the VALU instead of
// im2col + GEMM (which would pad each kernel position to 16 channels; such products are bound by
// their output bytes, not by the multiplies): a lane per output pixel over OG output channels, its
// taps gathered once (zero outside the input) and packed in pairs, each channel's sum by
// v_dot2_i32_i16 against the channel's pairs staged in LDS (read by every lane at one
// address).  The sum is int32 where that is exact -- the wrap path (the int32 wrap is its
// rule), or a channel whose bound sum |w| 2^15 + |bias| 2^8 stays below 2^31 -- and int64
// otherwise; then floor(acc / 2^8) clamped to [lo, hi] (saturation and a fused RELU / RELU6),
// as the GEMM path stores it.  w in the packed layout of cm_conv (ConvKernel.h:136-159).
constexpr uint32_t kCsMaxTaps = 80;          // taps a lane holds (40 pairs)
// taps x output channels up to which the VALU path beats the GEMM's (measured on MobileNetV2's
// 1x1 shapes: 32 x 192 at 28^2 pixels 18 vs 21 us, 64 x 384 at 14^2 21 vs 17 us)
constexpr uint64_t kCsMaxWork = 12288;
constexpr uint32_t kCsOg = 32;               // output channels a workgroup holds at most (4 at a time)

struct ConvSmall {
    const int16_t* x;
    const int16_t* w;
    const int16_t* bias;
    int16_t* y;
    uint32_t in_ch, in_h, in_w, out_ch, out_h, out_w, kh, kw, sh, sw, dh, dw, pt, pl;
    uint32_t per_m, tiles, last;             // the packed weights: entries per output channel, 16-channel
                                             // tiles, lanes of a position in the last tile
    uint32_t cs, cn, gs, wrap;
    int32_t lo, hi;
    uint32_t og;                             // output channels of a workgroup (a multiple of 4, <= kCsOg)
};

// PW: a pointwise convolution (1x1, stride 1, no padding, the output plane the input's): the
// lane's taps are its pixel in each input channel, loaded before the weights are staged.
template <uint32_t NP, bool PW>                // tap pairs, a multiple of 4 (16-byte LDS reads)
__global__ __launch_bounds__(256) void conv_small_kernel(ConvSmall c) {
    __shared__ __attribute__((aligned(16))) uint32_t wl[kCsOg][NP];
    __shared__ int32_t bl[kCsOg];
    __shared__ uint32_t exact[kCsOg], exact4[kCsOg / 4];
    __shared__ uint64_t ybase[kCsOg];         // a channel's offset in the output (the y pattern)
    const uint32_t t = threadIdx.x, plane = c.out_h * c.out_w, taps = c.in_ch * c.kh * c.kw, khw = c.kh * c.kw;
    const uint32_t oc0 = blockIdx.y * c.og, nb = blockIdx.z;
    const uint32_t og = min(c.og, c.out_ch - oc0);
    const int16_t* xb = c.x + (uint64_t)nb * c.in_ch * c.in_h * c.in_w;
    // the lane's output pixel and its taps, loaded before the weights are staged (their
    // latency under the staging's): PW from the input planes at the pixel; otherwise the taps
    // in order (ci, a, b) from running counters, the same for every lane (scalar registers),
    // so that all the loads go out at once
    const uint32_t p = blockIdx.x * 256 + t;
    const bool live = p < plane;
    uint32_t xv[NP];
    if constexpr (PW) {
#pragma unroll
        for (uint32_t pr = 0; pr < NP; pr++) {
            const uint32_t lo = live && 2 * pr < taps ? (uint32_t)(uint16_t)xb[(uint64_t)(2 * pr) * plane + p] : 0u;
            const uint32_t hi = live && 2 * pr + 1 < taps ? (uint32_t)(uint16_t)xb[(uint64_t)(2 * pr + 1) * plane + p] : 0u;
            xv[pr] = lo | (hi << 16);
        }
    } else {
        const uint32_t pc = live ? p : 0u;
        const uint32_t oh = pc / c.out_w, ow = pc - oh * c.out_w;
        const int ih0 = (int)(oh * c.sh) - (int)c.pt, iw0 = (int)(ow * c.sw) - (int)c.pl;
        // the kernel rows and columns whose input row / column lies inside the plane, as bit
        // masks (kh, kw <= 32), so that a tap's test is two shifts and an AND
        uint32_t rm = 0, cmk = 0;
        for (uint32_t a = 0; a < c.kh; a++) {
            const int ih = ih0 + (int)(a * c.dh);
            rm |= (ih >= 0 && ih < (int)c.in_h ? 1u : 0u) << a;
        }
        for (uint32_t b = 0; b < c.kw; b++) {
            const int iw = iw0 + (int)(b * c.dw);
            cmk |= (iw >= 0 && iw < (int)c.in_w ? 1u : 0u) << b;
        }
        if (!live) rm = 0;
        // the lane's offset from the window origin at row -pt, column -pl (never negative), and
        // the tap's offset from that origin, the same for every lane (scalar
        // registers, stepped as the counters run), so that a tap's load address is one add
        const uint32_t vo = oh * c.sh * c.in_w + ow * c.sw;
        int64_t uo = -((int64_t)c.pt * c.in_w + c.pl);
        const int64_t step_a = (int64_t)c.dh * c.in_w - (int64_t)c.kw * c.dw;
        const int64_t step_c = (int64_t)c.in_h * c.in_w - (int64_t)c.kh * c.dh * c.in_w;
        // the valid columns of the current kernel row, zero past the last input channel (the
        // taps past in_ch kh kw), updated only where a kernel row ends
        uint32_t ta = 0, tb = 0, ci = 0;
        uint32_t crow = (rm & 1u) ? cmk : 0u;
#pragma unroll
        for (uint32_t pr = 0; pr < NP; pr++) {
            uint32_t v2 = 0;
#pragma unroll
            for (uint32_t h = 0; h < 2; h++) {
                const bool in = (crow & (1u << tb)) != 0u;
                v2 |= (in ? (uint32_t)(uint16_t)xb[uo + (int64_t)vo] : 0u) << (16 * h);
                uo += c.dw;
                if (++tb == c.kw) {
                    tb = 0;
                    uo += step_a;
                    if (++ta == c.kh) {
                        ta = 0;
                        uo += step_c;
                        ci++;
                    }
                    crow = ci < c.in_ch && ((rm >> ta) & 1u) ? cmk : 0u;
                }
            }
            xv[pr] = v2;
        }
    }
    // the group's weights as int16 pairs in tap order (ci, a, b), zero past the taps
    for (uint32_t i = t; i < c.og * NP; i += 256) {
        const uint32_t o = i / NP, pr = i - o * NP;
        uint32_t v = 0;
#pragma unroll
        for (uint32_t h = 0; h < 2; h++) {
            const uint32_t tp = 2 * pr + h;
            if (o < og && tp < taps) {
                const uint32_t ci = tp / khw, pos = tp - ci * khw, ict = ci >> 4;
                const uint32_t lanes = ict + 1 == c.tiles ? c.last : 16u;
                v |= (uint32_t)(uint16_t)c.w[(uint64_t)(oc0 + o) * c.per_m + ict * khw * 16 + pos * lanes + (ci & 15)]
                     << (16 * h);
            }
        }
        wl[o][pr] = v;
    }
    if (t < kCsOg) bl[t] = t < og && c.bias ? (int32_t)c.bias[oc0 + t] : 0;
    __syncthreads();
    if (t < kCsOg) {
        // int32 is exact when sum |w| 2^15 + |bias| 2^8 < 2^31 (and always for the wrap rule)
        uint64_t bound = (uint64_t)(bl[t] < 0 ? -bl[t] : bl[t]) << 8;
        for (uint32_t pr = 0; pr < NP; pr++) {
            const int32_t w0 = (int16_t)(wl[t][pr] & 0xFFFF), w1 = (int16_t)(wl[t][pr] >> 16);
            bound += (uint64_t)((w0 < 0 ? -w0 : w0) + (w1 < 0 ? -w1 : w1)) << 15;
        }
        exact[t] = c.wrap || bound < ((uint64_t)1 << 31);
        const uint32_t oc = oc0 + t;
        ybase[t] = c.cn ? (uint64_t)(oc % c.cn) * c.cs + (uint64_t)(oc / c.cn) * c.gs : (uint64_t)oc * c.cs;
    }
    __syncthreads();
    if (t < kCsOg / 4) exact4[t] = exact[4 * t] & exact[4 * t + 1] & exact[4 * t + 2] & exact[4 * t + 3];
    __syncthreads();
    typedef short v2s __attribute__((ext_vector_type(2)));
    if (!live) return;                                    // no barrier follows
    int16_t* yb = c.y + (uint64_t)nb * c.out_ch * plane + p;
    // four channels at a time: four independent sums (channels past og have zero weights,
    // their stores are skipped)
    for (uint32_t o = 0; o < og; o += 4) {
        int64_t q[4];
        if (exact4[o / 4]) {
            int32_t acc[4];
#pragma unroll
            for (uint32_t j = 0; j < 4; j++) acc[j] = (int32_t)((uint32_t)bl[o + j] << 8);
#pragma unroll
            for (uint32_t pr = 0; pr < NP; pr += 4) {
#pragma unroll
                for (uint32_t j = 0; j < 4; j++) {
                    const uint4 wq = *reinterpret_cast<const uint4*>(&wl[o + j][pr]);
                    acc[j] = __builtin_amdgcn_sdot2(__builtin_bit_cast(v2s, xv[pr]), __builtin_bit_cast(v2s, wq.x), acc[j], false);
                    acc[j] = __builtin_amdgcn_sdot2(__builtin_bit_cast(v2s, xv[pr + 1]), __builtin_bit_cast(v2s, wq.y), acc[j], false);
                    acc[j] = __builtin_amdgcn_sdot2(__builtin_bit_cast(v2s, xv[pr + 2]), __builtin_bit_cast(v2s, wq.z), acc[j], false);
                    acc[j] = __builtin_amdgcn_sdot2(__builtin_bit_cast(v2s, xv[pr + 3]), __builtin_bit_cast(v2s, wq.w), acc[j], false);
                }
            }
#pragma unroll
            for (uint32_t j = 0; j < 4; j++) q[j] = acc[j] >> 8;
        } else {
#pragma unroll
            for (uint32_t j = 0; j < 4; j++) {
                long long acc = (long long)bl[o + j] * 256;
#pragma unroll
                for (uint32_t pr = 0; pr < NP; pr++) {
                    const uint32_t wv = wl[o + j][pr];
                    acc += (long long)(int16_t)(xv[pr] & 0xFFFF) * (int16_t)(wv & 0xFFFF) +
                           (long long)(int16_t)(xv[pr] >> 16) * (int16_t)(wv >> 16);
                }
                q[j] = acc >> 8;
            }
        }
#pragma unroll
        for (uint32_t j = 0; j < 4; j++)
            if (o + j < og) yb[ybase[o + j]] = (int16_t)(q[j] > c.hi ? c.hi : (q[j] < c.lo ? c.lo : q[j]));
    }
}

// ---------------------------------------------------------------- depthwise conv
__global__ __launch_bounds__(256) void conv_dw_kernel(const int16_t* __restrict__ x,
                                                      const int16_t* __restrict__ w,
                                                      const int16_t* __restrict__ bias,
                                                      int16_t* __restrict__ y, uint64_t total,
                                                      uint32_t ch, uint32_t in_h, uint32_t in_w,
                                                      uint32_t out_h, uint32_t out_w, uint32_t kh,
                                                      uint32_t kw, uint32_t sh, uint32_t sw,
                                                      uint32_t dh, uint32_t dw, uint32_t pt,
                                                      uint32_t pl, uint32_t dws, uint32_t cs,
                                                      uint32_t cn, uint32_t gs, uint32_t wrap, int32_t lo,
                                                      int32_t hi) {
    for (uint64_t o = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; o < total;
         o += (uint64_t)gridDim.x * blockDim.x) {
        const uint32_t ow = (uint32_t)(o % out_w);
        const uint64_t t1 = o / out_w;
        const uint32_t oh = (uint32_t)(t1 % out_h);
        const uint64_t t2 = t1 / out_h;
        const uint32_t c = (uint32_t)(t2 % ch);
        const uint64_t nb = t2 / ch;
        const int16_t* xp = x + (nb * ch + c) * in_h * in_w;
        const int16_t* wp = w + (uint64_t)c * dws;
        long long acc = bias ? (long long)bias[c] * 256 : 0;
        for (uint32_t a = 0; a < kh; a++) {
            const int ih = (int)(oh * sh + a * dh) - (int)pt;
            if (ih < 0 || ih >= (int)in_h) continue;
            for (uint32_t b = 0; b < kw; b++) {
                const int iw = (int)(ow * sw + b * dw) - (int)pl;
                if (iw < 0 || iw >= (int)in_w) continue;
                acc += (long long)xp[(uint64_t)ih * in_w + iw] * wp[a * kw + b];
            }
        }
        if (wrap) acc = (long long)(int32_t)(uint32_t)(unsigned long long)acc;
        long long q = acc >> 8;
        const uint64_t plane = (uint64_t)out_h * out_w;
        uint64_t base = cn ? (uint64_t)(c % cn) * cs + (uint64_t)(c / cn) * gs : (uint64_t)c * cs;
        y[nb * ch * plane + base + (uint64_t)oh * out_w + ow] = (int16_t)(q > hi ? hi : (q < lo ? lo : q));
    }
}

// Depthwise 3x3 stride 1 on rows of a multiple of 8 columns: a lane computes 8 columns x R
// rows.  Per input row it loads the 16-byte word of its 8 columns and the dwords either side
// (columns 8j - 2 .. 8j + 9, zero past the row), and every output takes its row's three
// taps as two v_dot2_i32_i16 against packed weight pairs, so no 16-bit value is unpacked.
// PL (the left pad, 0..2) fixes which pairs line up.  Sums are int32 where they are
// exact: the wrap path, or a channel whose bound sum |w| 2^15 + |bias| 2^8 stays below 2^31; int64 a value
// otherwise.
typedef short cm_s16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ int dot2(uint32_t x, uint32_t w, int acc) {
    return __builtin_amdgcn_sdot2(__builtin_bit_cast(cm_s16x2, x), __builtin_bit_cast(cm_s16x2, w), acc, false);
}

__device__ __forceinline__ uint32_t pack16(int lo, int hi) { return (uint32_t)(uint16_t)lo | ((uint32_t)hi << 16); }

template <int PL, int R>
__global__ __launch_bounds__(256) void conv_dw3v_kernel(const int16_t* __restrict__ x, const int16_t* __restrict__ w,
                                                        const int16_t* __restrict__ bias, int16_t* __restrict__ y,
                                                        uint32_t items, uint32_t strips, uint32_t groups, uint32_t ch,
                                                        uint32_t in_h, uint32_t in_w, uint32_t out_h, uint32_t out_w,
                                                        uint32_t pt, uint32_t dws, uint32_t cs, uint32_t cn,
                                                        uint32_t gs, uint32_t wrap, int32_t lo, int32_t hi) {
    const uint32_t per_plane = strips * groups;
    for (uint32_t it = blockIdx.x * blockDim.x + threadIdx.x; it < items; it += gridDim.x * blockDim.x) {
        const uint32_t p = it / per_plane, rem = it - p * per_plane;
        const uint32_t sidx = rem / groups, j = rem - sidx * groups;
        const uint32_t nb = p / ch, c = p - nb * ch;
        const int16_t* xp = x + (uint64_t)p * in_h * in_w;
        const int16_t* wp = w + (uint64_t)c * dws;
        int wv[9];
        uint32_t wabs = 0;
#pragma unroll
        for (int i = 0; i < 9; i++) {
            wv[i] = wp[i];
            wabs += (uint32_t)(wv[i] < 0 ? -wv[i] : wv[i]);
        }
        const int b0 = bias ? (int)bias[c] : 0;
        const uint64_t bound = (uint64_t)wabs * 32768u + (uint64_t)(b0 < 0 ? -b0 : b0) * 256u;
        const bool exact32 = wrap || bound < ((uint64_t)1 << 31);
        const int oh0 = (int)(sidx * R);
        const uint32_t c0 = 8 * j;                                   // first output column
        const uint64_t plane = (uint64_t)out_h * out_w;
        const uint64_t base = cn ? (uint64_t)(c % cn) * cs + (uint64_t)(c / cn) * gs : (uint64_t)c * cs;
        int16_t* yp = y + (uint64_t)nb * ch * plane + base + c0;
        if (!exact32) {
            // int64 per value (weights too large for an int32 bound): each tap loaded alone
            for (int i = 0; i < R && (uint32_t)(oh0 + i) < out_h; i++) {
#pragma unroll
                for (int t = 0; t < 8; t++) {
                    long long a64 = (long long)b0 * 256;
                    for (int a = 0; a < 3; a++) {
                        const int ih = oh0 + i - (int)pt + a;
                        if ((uint32_t)ih >= in_h) continue;
                        for (int b = 0; b < 3; b++) {
                            const int iw = (int)c0 + t - PL + b;
                            if ((uint32_t)iw < in_w) a64 += (long long)xp[(uint64_t)ih * in_w + iw] * wv[3 * a + b];
                        }
                    }
                    const long long v = a64 >> 8;
                    yp[(uint64_t)(oh0 + i) * out_w + t] = (int16_t)(v > hi ? hi : (v < lo ? lo : v));
                }
            }
            continue;
        }
        // weight pairs per kernel row: (w0, w1), (w2, 0) for an even first tap; (0, w0), (w1, w2) odd
        uint32_t wA[3], wB[3], wC[3], wD[3];
#pragma unroll
        for (int a = 0; a < 3; a++) {
            wA[a] = pack16(wv[3 * a], wv[3 * a + 1]);
            wB[a] = pack16(wv[3 * a + 2], 0);
            wC[a] = pack16(0, wv[3 * a]);
            wD[a] = pack16(wv[3 * a + 1], wv[3 * a + 2]);
        }
        int acc[R][8];
#pragma unroll
        for (int i = 0; i < R; i++)
#pragma unroll
            for (int t = 0; t < 8; t++) acc[i][t] = b0 * 256;
#pragma unroll
        for (int r = 0; r < R + 2; r++) {
            const int ih = oh0 - (int)pt + r;
            uint32_t W[6] = {0, 0, 0, 0, 0, 0};                      // columns c0 - 2 .. c0 + 9
            if ((uint32_t)ih < in_h) {
                const int16_t* xr = xp + (uint64_t)ih * in_w + c0;
                if (c0 + 8 <= in_w) {
                    const int4 mid = *reinterpret_cast<const int4*>(xr);
                    W[1] = (uint32_t)mid.x;
                    W[2] = (uint32_t)mid.y;
                    W[3] = (uint32_t)mid.z;
                    W[4] = (uint32_t)mid.w;
                }
                if (c0 >= 2) W[0] = *reinterpret_cast<const uint32_t*>(xr - 2);
                if (c0 + 10 <= in_w) W[5] = *reinterpret_cast<const uint32_t*>(xr + 8);
            }
#pragma unroll
            for (int a = 0; a < 3; a++) {
                const int i = r - a;                                   // the output row fed at tap row a
                if (i < 0 || i >= R) continue;
#pragma unroll
                for (int t = 0; t < 8; t++) {
                    const int q0 = t - PL + 2;                         // window index of tap b = 0
                    if ((q0 & 1) == 0) {
                        acc[i][t] = dot2(W[q0 >> 1], wA[a], acc[i][t]);
                        acc[i][t] = dot2(W[(q0 >> 1) + 1], wB[a], acc[i][t]);
                    } else {
                        acc[i][t] = dot2(W[q0 >> 1], wC[a], acc[i][t]);
                        acc[i][t] = dot2(W[(q0 >> 1) + 1], wD[a], acc[i][t]);
                    }
                }
            }
        }
#pragma unroll
        for (int i = 0; i < R; i++) {
            if ((uint32_t)(oh0 + i) >= out_h) break;
            int q[8];
#pragma unroll
            for (int t = 0; t < 8; t++) q[t] = clamp_i32(acc[i][t] >> 8, lo, hi);
            int4 o;
            o.x = __builtin_bit_cast(int, __builtin_amdgcn_cvt_pk_i16(q[0], q[1]));
            o.y = __builtin_bit_cast(int, __builtin_amdgcn_cvt_pk_i16(q[2], q[3]));
            o.z = __builtin_bit_cast(int, __builtin_amdgcn_cvt_pk_i16(q[4], q[5]));
            o.w = __builtin_bit_cast(int, __builtin_amdgcn_cvt_pk_i16(q[6], q[7]));
            store_stream(yp + (uint64_t)(oh0 + i) * out_w, o);
        }
    }
}

// Depthwise 3x3, dilation 1, stride S both ways, over so few columns that the launch is its latency, or
// over the narrowest rows: each lane computes R output rows of one column (a vertical strip) from the (R - 1) S + 3 input rows' three
// taps, a load a tap with no edge to mend.  One workgroup a unit or fewer, us (conv_dw3_kernel): one
// image of 96 channels at 14 x 14, stride 2 3.9 (4.3), of 960 at 7 x 7 4.0 (4.25), 32 images of 32 at 3 x 3 3.8
// (5.3).  Sums as conv_dw3v_kernel.
template <int S, int R>
__global__ __launch_bounds__(256) void conv_dw3_strip_kernel(const int16_t* __restrict__ x, const int16_t* __restrict__ w,
                                                             const int16_t* __restrict__ bias, int16_t* __restrict__ y,
                                                             uint32_t items, uint32_t strips, uint32_t ch,
                                                             uint32_t in_h, uint32_t in_w, uint32_t out_h,
                                                             uint32_t out_w, uint32_t pt, uint32_t pl, uint32_t dws,
                                                             uint32_t cs, uint32_t cn, uint32_t gs, uint32_t wrap,
                                                             int32_t lo, int32_t hi) {
    constexpr int NR = (R - 1) * S + 3;
    const uint32_t per_plane = strips * out_w;
    for (uint32_t it = blockIdx.x * blockDim.x + threadIdx.x; it < items; it += gridDim.x * blockDim.x) {
        const uint32_t p = it / per_plane, rem = it - p * per_plane;
        const uint32_t sidx = rem / out_w, ow = rem - sidx * out_w;
        const uint32_t nb = p / ch, c = p - nb * ch;
        const int16_t* xp = x + (uint64_t)p * in_h * in_w;
        const int16_t* wp = w + (uint64_t)c * dws;
        int wv[9];
        uint32_t wabs = 0;
#pragma unroll
        for (int i = 0; i < 9; i++) {
            wv[i] = wp[i];
            wabs += (uint32_t)(wv[i] < 0 ? -wv[i] : wv[i]);
        }
        const int b0 = bias ? (int)bias[c] : 0;
        const int oh0 = (int)(sidx * R);
        const int ih0 = oh0 * S - (int)pt, iw0 = (int)(ow * S) - (int)pl;
        bool cv[3];
#pragma unroll
        for (int b = 0; b < 3; b++) cv[b] = (uint32_t)(iw0 + b) < in_w;
        int v[NR][3];
#pragma unroll
        for (int r = 0; r < NR; r++) {
            const int ih = ih0 + r;
            const bool rv = (uint32_t)ih < in_h;
            const int16_t* xr = xp + (int64_t)ih * in_w + iw0;
#pragma unroll
            for (int b = 0; b < 3; b++) v[r][b] = (rv && cv[b]) ? (int)xr[b] : 0;
        }
        const uint64_t bound = (uint64_t)wabs * 32768u + (uint64_t)(b0 < 0 ? -b0 : b0) * 256u;
        int out[R];
        if (wrap || bound < ((uint64_t)1 << 31)) {
#pragma unroll
            for (int i = 0; i < R; i++) {
                uint32_t acc = (uint32_t)b0 << 8;
#pragma unroll
                for (int a = 0; a < 3; a++)
#pragma unroll
                    for (int b = 0; b < 3; b++) acc += (uint32_t)(v[i * S + a][b] * wv[a * 3 + b]);
                out[i] = clamp_i32((int)acc >> 8, lo, hi);
            }
        } else {
#pragma unroll
            for (int i = 0; i < R; i++) {
                long long acc = (long long)b0 * 256;
#pragma unroll
                for (int a = 0; a < 3; a++)
#pragma unroll
                    for (int b = 0; b < 3; b++) acc += (long long)v[i * S + a][b] * wv[a * 3 + b];
                const long long q = acc >> 8;
                out[i] = (int)(q > hi ? hi : (q < lo ? lo : q));
            }
        }
        const uint64_t plane = (uint64_t)out_h * out_w;
        const uint64_t base = cn ? (uint64_t)(c % cn) * cs + (uint64_t)(c / cn) * gs : (uint64_t)c * cs;
        int16_t* yp = y + (uint64_t)nb * ch * plane + base + ow;
#pragma unroll
        for (int i = 0; i < R; i++)
            if ((uint32_t)(oh0 + i) < out_h) yp[(uint64_t)(oh0 + i) * out_w] = (int16_t)out[i];
    }
}

// Depthwise 3x3, dilation 1, stride S both ways, at any width (the MobileNet blocks): a lane computes R rows
// of 8 / S output columns from the 10 input columns 8 j - pad_left .. + 9 of every input row, loaded as 20
// bytes at any alignment.  A load a tap kept the address unit busy: 27 two-byte loads for 4 outputs at
// stride 2, 96 channels at 32 x 112 x 112 36.7 us, 20.7 this way (96 MB: 16.1 at 6 TB/s); 384 at 14 x 14
// 7.1 and 5.4, 960 at 7 x 7 6.2 and 5.3.  Columns outside the plane are masked off; at the tensor's ends
// the words move inside it and are shifted back.  Two rows: a longer strip saves loads where the planes
// are large (20.0) but its code and its chain cost the small ones (4 rows: 384 at 14 x 14 7.0, one image
// 4.5 against 3.5).  Rows of a multiple of 8 columns at stride 1 keep the aligned words above (144 channels
// at 32 x 56 x 56 14.6 us, 18.6 here).  Taps and sums as conv_dw3v_kernel.
template <int S, int R>
__global__ __launch_bounds__(256) void conv_dw3_kernel(const int16_t* __restrict__ x, const int16_t* __restrict__ w,
                                                       const int16_t* __restrict__ bias, int16_t* __restrict__ y,
                                                       uint32_t items, uint32_t planes, uint32_t strips, uint32_t groups,
                                                       uint32_t ch, uint32_t in_h, uint32_t in_w, uint32_t out_h,
                                                       uint32_t out_w, uint32_t pt, uint32_t pl, uint32_t dws, uint32_t cs,
                                                       uint32_t cn, uint32_t gs, uint32_t wrap, int32_t lo, int32_t hi) {
    constexpr int T = 8 / S;                                         // output columns of a lane
    const uint32_t per_plane = strips * groups, in_hw = in_h * in_w;
    for (uint32_t it = blockIdx.x * blockDim.x + threadIdx.x; it < items; it += gridDim.x * blockDim.x) {
        const uint32_t p = it / per_plane, rem = it - p * per_plane;
        const uint32_t sidx = rem / groups, j = rem - sidx * groups;
        const uint32_t nb = p / ch, c = p - nb * ch;
        const int16_t* xp = x + (uint64_t)p * in_hw;
        const int16_t* wp = w + (uint64_t)c * dws;
        // the last lane of a row ends at the row's end (columns of the lane before it come out twice, the same)
        const int oh0 = (int)(sidx * R), ow0 = (int)min(T * j, out_w - min((uint32_t)T, out_w));
        const int ih0 = oh0 * S - (int)pt, iw0 = ow0 * S - (int)pl;
        // the plane offsets at which the words of 10 columns stay inside the tensor (of 10 elements or more)
        const int first = -(int)min((uint64_t)p * in_hw, (uint64_t)1 << 29);
        const int last = (int)min((uint64_t)(planes - p) * in_hw, (uint64_t)1 << 30) - 10;
        constexpr int NR = (R - 1) * S + 3;
        uint32_t v[NR][5];
        auto offset = [&](int r) { return min(max(ih0 + r, 0), (int)in_h - 1) * (int)in_w + iw0; };
        int moved = 0;
#pragma unroll
        for (int r = 0; r < NR; r++) {
            const int o = offset(r), at = min(max(o, first), last);
            moved = max(moved, max(o - at, at - o));
            __builtin_memcpy(v[r], xp + at, 16);
            __builtin_memcpy(v[r] + 4, xp + at + 8, 4);
        }
        int wv[9];
        uint32_t wabs = 0;
#pragma unroll
        for (int i = 0; i < 9; i++) {
            wv[i] = wp[i];
            wabs += (uint32_t)(wv[i] < 0 ? -wv[i] : wv[i]);
        }
        const int b0 = bias ? (int)bias[c] : 0;
        const uint64_t bound = (uint64_t)wabs * 32768u + (uint64_t)(b0 < 0 ? -b0 : b0) * 256u;
        if (moved > 0) {
            // at the tensor's ends: the words back to their columns, one element at a time (what comes in
            // lies outside the plane and is masked below)
#pragma unroll 1
            for (int n = 0; n < min(moved, 10); n++) {
#pragma unroll
                for (int r = 0; r < NR; r++) {
                    const int d = offset(r) - min(max(offset(r), first), last);
                    if (d > n) {
#pragma unroll
                        for (int k = 0; k < 5; k++) v[r][k] = __builtin_amdgcn_alignbit(k < 4 ? v[r][k + 1 < 5 ? k + 1 : 4] : 0u, v[r][k], 16);
                    } else if (-d > n) {
#pragma unroll
                        for (int k = 4; k >= 0; k--) v[r][k] = __builtin_amdgcn_alignbit(v[r][k], k > 0 ? v[r][k - 1 > 0 ? k - 1 : 0] : 0u, 16);
                    }
                }
            }
        }
        uint32_t m[5];
#pragma unroll
        for (int k = 0; k < 5; k++)
            m[k] = ((uint32_t)(iw0 + 2 * k) < in_w ? 0xFFFFu : 0u) | ((uint32_t)(iw0 + 2 * k + 1) < in_w ? 0xFFFF0000u : 0u);
#pragma unroll
        for (int r = 0; r < NR; r++) {
            const bool in = (uint32_t)(ih0 + r) < in_h;
#pragma unroll
            for (int k = 0; k < 5; k++) v[r][k] &= in ? m[k] : 0u;
        }
        const uint64_t plane = (uint64_t)out_h * out_w;
        const uint64_t base = cn ? (uint64_t)(c % cn) * cs + (uint64_t)(c / cn) * gs : (uint64_t)c * cs;
        int16_t* yp = y + (uint64_t)nb * ch * plane + base + ow0;
        const int nv = (int)min(out_w, (uint32_t)T);                 // the columns inside
        int q[R][T];                                                 // floor(acc / 2^8): within 26 bits
        if (!wrap && bound >= ((uint64_t)1 << 31)) {
            // weights too large for an int32 bound: int64 a value, from the same words (32 images of 384 channels,
            // 29 x 29 stride 1, 56 x 56 stride 2: 19.4 and 28.1 us; with every tap loaded alone 135.7 and 124.6)
#pragma unroll
            for (int i = 0; i < R; i++)
#pragma unroll
                for (int t = 0; t < T; t++) {
                    long long acc = (long long)b0 * 256;
#pragma unroll
                    for (int k = 0; k < 9; k++) {
                        const int col = t * S + k % 3;
                        const uint32_t u = v[i * S + k / 3][col >> 1];
                        acc += (long long)((col & 1) ? (int)u >> 16 : (int)(int16_t)u) * wv[k];
                    }
                    q[i][t] = (int)(acc >> 8);
                }
        } else {
#pragma unroll
            for (int i = 0; i < R; i++)
#pragma unroll
                for (int t = 0; t < T; t++) {
                    int acc = b0 * 256;
#pragma unroll
                    for (int a = 0; a < 3; a++) {
                        const uint32_t* vr = v[i * S + a];
                        // weight pairs for an even first column (w0, w1), (w2, 0), an odd one (0, w0), (w1, w2)
                        if ((t * S & 1) == 0) {
                            acc = dot2(vr[t * S >> 1], pack16(wv[3 * a], wv[3 * a + 1]), acc);
                            acc = dot2(vr[(t * S >> 1) + 1], pack16(wv[3 * a + 2], 0), acc);
                        } else {
                            acc = dot2(vr[t * S >> 1], pack16(0, wv[3 * a]), acc);
                            acc = dot2(vr[(t * S >> 1) + 1], pack16(wv[3 * a + 1], wv[3 * a + 2]), acc);
                        }
                    }
                    q[i][t] = acc >> 8;
                }
        }
#pragma unroll
        for (int i = 0; i < R; i++) {
            if ((uint32_t)(oh0 + i) >= out_h) break;
            uint32_t o[T / 2];
#pragma unroll
            for (int t = 0; t < T; t += 2)
                o[t / 2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pk_i16(clamp_i32(q[i][t], lo, hi), clamp_i32(q[i][t + 1], lo, hi)));
            int16_t* dst = yp + (uint64_t)(oh0 + i) * out_w;
            if (nv == T) {
                __builtin_memcpy(dst, o, 2 * T);
            } else {
#pragma unroll
                for (int t = 0; t < T - 1; t += 2) {
                    if (t + 1 < nv) __builtin_memcpy(dst + t, &o[t / 2], 4);
                    else if (t < nv) dst[t] = (int16_t)o[t / 2];
                }
            }
        }
    }
}

// ---------------------------------------------------------------- skinny products (int32 wrap)
// C = sat16(wrap32(A . B) >> 8) for A of at most 32 rows: the decode step's linears, where a
// 128-column MFMA tile would be mostly padding and the plane split would cost more than the
// product.  The wrap rule makes the int32 sum mod 2^32 exact in any order, so v_dot2_i32_i16
// (two products per lane-op, no clamp) accumulates it directly and split k needs no care.
// A wavefront takes 128 columns (a pair per lane) and one slice of kSkinnyKc k; A's rows of
// the slice sit in LDS as k pairs, read as broadcasts.  B layouts (BL): 0 row-major [k][m]
// and 1 the packed 32-column tiles (one 4-byte load per k row for the lane's two columns,
// paired by byte permutes); 2 transposed [m][k] (a column's k contiguous: 16-byte loads of
// 8 k).  Every B load of the slice is issued before the first product.  With several slices
// each wavefront writes its int32 partials [slice][ks][n][m] for skinny_reduce_kernel.
constexpr uint32_t kSkinnyKc = 64;
constexpr uint32_t kSkinnySegs = 4;

// The products of one skinny launch: up to kSkinnySegs B / C / m over the same A rows (batch 1),
// or one product over `batch` slices.  Segment s owns column blocks [cb0[s], cb0[s + 1]) of
// the grid and output pairs [pair0[s], pair0[s + 1]) of the reduce.
struct SkinnySegs {
    const int16_t* b[kSkinnySegs];
    int16_t* c[kSkinnySegs];
    int32_t* part[kSkinnySegs];
    uint32_t m[kSkinnySegs], cb0[kSkinnySegs];
    uint64_t pair0[kSkinnySegs];
    uint32_t count;
};

template <int NR, int BL>
__global__ __launch_bounds__(64) void skinny_wrap_kernel(const int16_t* __restrict__ a, uint64_t a_bs,
                                                          SkinnySegs segs, uint64_t b_bs, uint64_t c_bs, uint32_t n,
                                                          uint32_t k) {
    constexpr uint32_t KP = kSkinnyKc / 2;                                // k pairs per slice
    __shared__ __attribute__((aligned(16))) uint32_t sa[NR][KP];
    uint32_t si = 0;                                                      // this workgroup's segment
    for (uint32_t i = 1; i < segs.count; i++)
        if (blockIdx.x >= segs.cb0[i]) si = i;
    const int16_t* __restrict__ b = segs.b[si];
    int16_t* __restrict__ c = segs.c[si];
    int32_t* __restrict__ part = segs.part[si];
    const uint32_t m = segs.m[si];
    const uint32_t lane = threadIdx.x, cb = blockIdx.x - segs.cb0[si], ks = blockIdx.y, bt = blockIdx.z,
                   nks = gridDim.y;
    const uint32_t k0 = ks * kSkinnyKc, k1 = min(k, k0 + kSkinnyKc);
    const int16_t* ab = a + bt * a_bs;
    const int16_t* bb = b + bt * b_bs;
    const uint32_t j0 = cb * 128 + 2 * lane;
    const bool live = j0 < m;
    // B's pairs (B[kk][j], B[kk+1][j]) of the slice for columns j0 and j0 + 1
    uint32_t p0[KP], p1[KP];
    if (BL == 2) {
#pragma unroll
        for (uint32_t q = 0; q < KP / 4; q++) {
            const uint32_t kk = k0 + 8 * q;
            int4 x = make_int4(0, 0, 0, 0), y = make_int4(0, 0, 0, 0);
            if (live && kk < k1) {                          // k1 - k0 is a multiple of 8 here
                x = *reinterpret_cast<const int4*>(bb + (uint64_t)j0 * k + kk);
                y = *reinterpret_cast<const int4*>(bb + (uint64_t)(j0 + 1) * k + kk);
            }
            p0[4 * q] = x.x; p0[4 * q + 1] = x.y; p0[4 * q + 2] = x.z; p0[4 * q + 3] = x.w;
            p1[4 * q] = y.x; p1[4 * q + 1] = y.y; p1[4 * q + 2] = y.z; p1[4 * q + 3] = y.w;
        }
    } else {
#pragma unroll
        for (uint32_t i = 0; i < KP; i++) {
            const uint32_t kk = k0 + 2 * i;
            uint32_t w0 = 0, w1 = 0;
            if (live && kk < k1) {                          // k1 - k0 is even
                const uint64_t o0 = BL == 1 ? ((uint64_t)(j0 >> 5) * k + kk) * 32 + (j0 & 31) : (uint64_t)kk * m + j0;
                const uint64_t o1 = BL == 1 ? o0 + 32 : o0 + m;
                w0 = *reinterpret_cast<const uint32_t*>(bb + o0);
                w1 = *reinterpret_cast<const uint32_t*>(bb + o1);
            }
            p0[i] = __builtin_amdgcn_perm(w1, w0, 0x05040100u);
            p1[i] = __builtin_amdgcn_perm(w1, w0, 0x07060302u);
        }
    }
    // A's rows of the slice (zero past n and past k)
    for (uint32_t e = lane; e < NR * KP; e += 64) {
        const uint32_t r = e / KP, kk = k0 + 2 * (e - r * KP);
        sa[r][e - r * KP] = (r < n && kk < k1) ? *reinterpret_cast<const uint32_t*>(ab + (uint64_t)r * k + kk) : 0u;
    }
    __syncthreads();
    typedef short v2s __attribute__((ext_vector_type(2)));
    int acc0[NR], acc1[NR];
#pragma unroll
    for (int r = 0; r < NR; r++) acc0[r] = acc1[r] = 0;
#pragma unroll
    for (uint32_t i = 0; i < KP; i += 4) {
#pragma unroll
        for (int r = 0; r < NR; r++) {
            const uint4 av = *reinterpret_cast<const uint4*>(&sa[r][i]);
            const uint32_t a4[4] = {av.x, av.y, av.z, av.w};
#pragma unroll
            for (int t = 0; t < 4; t++) {
                acc0[r] = __builtin_amdgcn_sdot2(__builtin_bit_cast(v2s, a4[t]), __builtin_bit_cast(v2s, p0[i + t]),
                                                 acc0[r], false);
                acc1[r] = __builtin_amdgcn_sdot2(__builtin_bit_cast(v2s, a4[t]), __builtin_bit_cast(v2s, p1[i + t]),
                                                 acc1[r], false);
            }
        }
    }
    int16_t* cbt = c + bt * c_bs;
    auto store = [&](uint32_t r, int s0, int s1) {
        const int q0 = min(max(s0 >> 8, -32768), 32767), q1 = min(max(s1 >> 8, -32768), 32767);
        *reinterpret_cast<uint32_t*>(cbt + (uint64_t)r * m + j0) = (uint32_t)(uint16_t)q0 | ((uint32_t)q1 << 16);
    };
    if (nks == 1) {
        if (live) {
#pragma unroll
            for (int r = 0; r < NR; r++)
                if ((uint32_t)r < n) store(r, acc0[r], acc1[r]);
        }
        return;
    }
    if (!live) return;
    const uint64_t per = (uint64_t)n * m;
    int32_t* pp = part + ((uint64_t)bt * nks + ks) * per;
#pragma unroll
    for (int r = 0; r < NR; r++)
        if ((uint32_t)r < n) *reinterpret_cast<int2*>(pp + (uint64_t)r * m + j0) = make_int2(acc0[r], acc1[r]);
}

// Sums the int32 partials of the k slices (wrapping) and applies the output rule: a lane per
// pair of outputs.
__global__ __launch_bounds__(256) void skinny_reduce_kernel(SkinnySegs segs, uint64_t c_bs, uint32_t n,
                                                            uint32_t nks, uint32_t batch, uint64_t total) {
    for (uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += (uint64_t)gridDim.x * blockDim.x) {
        uint32_t si = 0;
        for (uint32_t j = 1; j < segs.count; j++)
            if (e >= segs.pair0[j]) si = j;
        const uint64_t per = (uint64_t)n * segs.m[si], pairs = per / 2, el = e - segs.pair0[si];
        const uint64_t bt = el / pairs, i = 2 * (el - bt * pairs);
        int16_t* c = segs.c[si];
        const int32_t* pp = segs.part[si] + bt * nks * per + i;
        uint32_t s0 = 0, s1 = 0;
        uint32_t q = 0;
        for (; q + 8 <= nks; q += 8) {                 // eight slices' loads in flight at once
            int2 v[8];
#pragma unroll
            for (int u = 0; u < 8; u++) v[u] = *reinterpret_cast<const int2*>(pp + (uint64_t)(q + u) * per);
#pragma unroll
            for (int u = 0; u < 8; u++) {
                s0 += (uint32_t)v[u].x;
                s1 += (uint32_t)v[u].y;
            }
        }
        for (; q < nks; q++) {
            const int2 v = *reinterpret_cast<const int2*>(pp + (uint64_t)q * per);
            s0 += (uint32_t)v.x;
            s1 += (uint32_t)v.y;
        }
        const int q0 = min(max((int)s0 >> 8, -32768), 32767), q1 = min(max((int)s1 >> 8, -32768), 32767);
        *reinterpret_cast<uint32_t*>(c + bt * c_bs + i) = (uint32_t)(uint16_t)q0 | ((uint32_t)q1 << 16);
    }
}

// ---------------------------------------------------------------- skinny products on split weights
// C = sat16(wrap32(A . B) >> 8) for A of at most 16 rows against a weight already split into
// byte planes (cm_matmul_split_b).  Sixteen rows are exactly one v_mfma_i32_16x16x64_i8
// operand, so the products run on MFMA over limbs with the plane GEMM's recombination, and a
// workgroup owns NB 16-column blocks for the whole k: its W wavefronts take the 64-k steps w,
// w + W, .. (the loads of a chunk of sp_chunk(NB) steps all in flight before the chunk's products)
// and add their wrapped partials in LDS, so there are no partial buffers and no second launch.
// A is split in registers, 16 k of row l % 16 per lane (the MFMA operand layout), its row sums
// taken on the way; B's column sums come from the plane image.  Everything the stores of a
// thread's first kSpPre output elements read besides the product (B's column sums, the output
// job's parameter entry and x) is loaded before the products, under the weight loads.  NB
// trades the workgroups a weight's columns give (one MFMA block each: narrow weights) against
// the A rows every workgroup reads again (wide ones).
// 64-k steps whose loads a wavefront issues together, wavefronts of an NB-block workgroup (the
// register budget of its launch bounds), and the output elements a thread prefetches for
__host__ __device__ constexpr uint32_t sp_chunk(uint32_t nb) { return nb == 4 ? 2u : 4u; }
__host__ __device__ constexpr uint32_t sp_max_waves(uint32_t nb) { return nb == 1 ? 16u : 8u; }
__host__ __device__ constexpr uint32_t sp_pre(uint32_t nb) { return nb == 1 ? 1u : 2u; }

struct SkinnyPlaneSegs {
    const int8_t* hi[kSkinnySegs];
    const int8_t* lo[kSkinnySegs];
    const int32_t* part[kSkinnySegs];
    int16_t* c[kSkinnySegs];
    uint32_t m[kSkinnySegs], lines_p[kSkinnySegs], cb0[kSkinnySegs];
    uint32_t count;
};

// A row-ops COPY / ADDX job applied to a one-product launch's output as it is stored: out[r][j]
// = copy_addx(x[r][j], C[r][j]) with the job's op word (A kind, output kind, flags), its
// parameter block and bq_sh (the residual add of a decode linear); out == nullptr: none.
struct SkinnyAddx {
    const uint8_t* x;
    uint8_t* out;
    const uint8_t* params;
    uint32_t op, bq_sh;
};

// The operands of one output element's store other than the product, as loaded (nothing
// waits for them before the weight loads go out): B's column sums of the first kSpSlabs slabs,
// the output job's parameter entry and x (int16 or int32).
constexpr uint32_t kSpSlabs = 4;
struct SkinnyEpiIn {
    uint32_t cs[kSpSlabs] = {0, 0, 0, 0};
    uint4 prm{};
    int32_t x = 0;
};

// The wrapped partial products of one skinny workgroup: NB 16-column blocks whose plane lines
// start at bh[b] / bl[b] (the block's first column), into red [W][16][16 NB] and A's row sums
// into rsum [W][16]; ends with the workgroup barrier.  SAT: each wavefront's three limb sums
// (exact in int32) into red [3][W][16][16 NB] -- HH, MID, LL -- for the exact recombination.
template <uint32_t NB, bool SAT = false>
__device__ __forceinline__ void skinny_products(const int16_t* __restrict__ a, uint32_t n, uint32_t k, uint32_t kp,
                                                const int8_t* const (&bh)[NB], const int8_t* const (&bl)[NB],
                                                uint32_t* red, int32_t* rsum) {
    constexpr uint32_t COLS = 16 * NB, CH = sp_chunk(NB);
    const uint32_t W = blockDim.x >> 6, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const uint32_t r = lane & 15, g = lane >> 4;             // A row and B column of a block; k group
    const uint32_t nsteps = kp / 64;
    const bool row_ok = r < n;
    const int16_t* arow = a + (uint64_t)(row_ok ? r : 0) * k;
    const int4 pad8 = make_int4(0x00800080, 0x00800080, 0x00800080, 0x00800080);   // eight kPad: A' = 0
    v4i hh[NB], mid[NB], ll[NB];
#pragma unroll
    for (uint32_t b = 0; b < NB; b++) hh[b] = mid[b] = ll[b] = v4i{0, 0, 0, 0};
    int32_t asum = 0;
    for (uint32_t s0 = wave; s0 < nsteps; s0 += W * CH) {
        int4 av[CH][2];
        v4i bhv[CH][NB], blv[CH][NB];
#pragma unroll
        for (uint32_t u = 0; u < CH; u++) {
            const uint32_t st = s0 + u * W;
            const bool live = st < nsteps;
            const uint32_t kk = (live ? st : 0) * 64 + 16 * g;
            // k % 8 == 0: each half of the lane's 16 k is wholly real or wholly past k; a half past
            // k loads row 0's first 8 (in bounds) and takes the pad instead
            const bool h0 = live && row_ok && kk + 8 <= k, h1 = live && row_ok && kk + 16 <= k;
            const int4 a0 = *reinterpret_cast<const int4*>(arow + (h0 ? kk : 0));
            const int4 a1 = *reinterpret_cast<const int4*>(arow + (h1 ? kk + 8 : 0));
            av[u][0] = h0 ? a0 : pad8;
            av[u][1] = h1 ? a1 : pad8;
#pragma unroll
            for (uint32_t b = 0; b < NB; b++) {
                const uint64_t off = (uint64_t)r * kp + kk;
                bhv[u][b] = *reinterpret_cast<const v4i*>(bh[b] + off);
                blv[u][b] = *reinterpret_cast<const v4i*>(bl[b] + off);
            }
        }
#pragma unroll
        for (uint32_t u = 0; u < CH; u++) {
            if (s0 + u * W >= nsteps) break;                  // wave-uniform
            const uint32_t kk = (s0 + u * W) * 64 + 16 * g;
            if (row_ok && kk + 8 <= k) asum += sum8(av[u][0]);
            if (row_ok && kk + 16 <= k) asum += sum8(av[u][1]);
            uint2 h0, l0, h1, l1;
            split8(av[u][0], h0, l0);
            split8(av[u][1], h1, l1);
            const v4i ah{(int)h0.x, (int)h0.y, (int)h1.x, (int)h1.y}, al{(int)l0.x, (int)l0.y, (int)l1.x, (int)l1.y};
#pragma unroll
            for (uint32_t b = 0; b < NB; b++) hh[b] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ah, bhv[u][b], hh[b], 0, 0, 0);
#pragma unroll
            for (uint32_t b = 0; b < NB; b++) mid[b] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ah, blv[u][b], mid[b], 0, 0, 0);
#pragma unroll
            for (uint32_t b = 0; b < NB; b++) ll[b] = __builtin_amdgcn_mfma_i32_16x16x64_i8(al, blv[u][b], ll[b], 0, 0, 0);
#pragma unroll
            for (uint32_t b = 0; b < NB; b++) mid[b] = __builtin_amdgcn_mfma_i32_16x16x64_i8(al, bhv[u][b], mid[b], 0, 0, 0);
        }
    }
    // this wavefront's wrapped partials: lane l holds column l % 16 of each block, rows 4 g .. + 3
#pragma unroll
    for (uint32_t b = 0; b < NB; b++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t e = (wave * 16 + 4 * g + i) * COLS + 16 * b + r;
            if constexpr (SAT) {
                const uint32_t plane = W * 16 * COLS;
                red[e] = (uint32_t)hh[b][i];
                red[plane + e] = (uint32_t)mid[b][i];
                red[2 * plane + e] = (uint32_t)ll[b][i];
            } else {
                red[e] = ((uint32_t)hh[b][i] << 16) + ((uint32_t)mid[b][i] << 8) + (uint32_t)ll[b][i];
            }
        }
    asum += __shfl_xor(asum, 16, 64);
    asum += __shfl_xor(asum, 32, 64);
    if (g == 0) rsum[wave * 16 + r] = asum;
    __syncthreads();
}

// C[row][col] of a skinny workgroup from its wavefronts' partials (column cl of the tile), A's
// row sums and B's column sum cs.
__device__ __forceinline__ int16_t skinny_value(const uint32_t* red, const int32_t* rsum, uint32_t W, uint32_t cols,
                                                uint32_t row, uint32_t cl, uint32_t k, uint32_t cs) {
    uint32_t acc = 0u - 16384u * k, rs = 0;
    for (uint32_t w = 0; w < W; w++) {
        acc += red[(w * 16 + row) * cols + cl];
        rs += (uint32_t)rsum[w * 16 + row];
    }
    acc += 128u * rs + 128u * cs;
    return (int16_t)min(max((int32_t)acc >> 8, -32768), 32767);
}

// The same by the saturating rule: the wavefronts' limb sums (red [3][W][16][cols]) and the
// row / column sums recombined exactly in int64 (each term is exact in int32: |A|, |B| <=
// 2^15 and k <= 32768), then floor(acc / 2^8) saturated to int16.
__device__ __forceinline__ int16_t skinny_value_sat(const uint32_t* red, const int32_t* rsum, uint32_t W,
                                                    uint32_t cols, uint32_t row, uint32_t cl, uint32_t k,
                                                    uint32_t cs) {
    const uint32_t plane = W * 16 * cols;
    long long acc = -16384ll * k, rs = 0;
    for (uint32_t w = 0; w < W; w++) {
        const uint32_t e = (w * 16 + row) * cols + cl;
        acc += ((long long)(int32_t)red[e] << 16) + ((long long)(int32_t)red[plane + e] << 8) +
               (long long)(int32_t)red[2 * plane + e];
        rs += rsum[w * 16 + row];
    }
    acc += 128ll * rs + 128ll * (int32_t)cs;
    const long long q = acc >> 8;
    return (int16_t)(q > 32767 ? 32767 : (q < -32768 ? -32768 : q));
}

// B's column sum of column col from the slabs a prefetch took (the first kSpSlabs) and the rest.
__device__ __forceinline__ uint32_t skinny_colsum(const uint32_t (&pre)[kSpSlabs], const int32_t* part, uint32_t nslab,
                                                  uint32_t lp, uint32_t col) {
    uint32_t cs = 0;
#pragma unroll
    for (uint32_t sl = 0; sl < kSpSlabs; sl++) cs += pre[sl];
    for (uint32_t sl = kSpSlabs; sl < nslab; sl++) cs += (uint32_t)part[(uint64_t)sl * lp + col];
    return cs;
}

// XK: the output job's x kind (0: no job, 1: int16, 2: int32); SAT: the saturating rule (no job).
template <uint32_t NB, uint32_t XK, bool SAT = false>
__global__ __launch_bounds__(64 * sp_max_waves(NB)) void skinny_planes_kernel(const int16_t* __restrict__ a, uint32_t n,
                                                                       uint32_t k, uint32_t kp, uint32_t nslab,
                                                                       SkinnyPlaneSegs segs, SkinnyAddx ax) {
    constexpr uint32_t COLS = 16 * NB;
    extern __shared__ __attribute__((aligned(16))) uint32_t sp_lds[];
    const uint32_t W = blockDim.x >> 6;
    static_assert(!SAT || XK == 0, "no output job on the saturating products");
    uint32_t* red = sp_lds;                                  // [W][16][COLS] wrapped partials ([3][..] SAT)
    int32_t* rsum = reinterpret_cast<int32_t*>(sp_lds + (SAT ? 3 : 1) * W * 16 * COLS);   // [W][16] A row sums
    uint32_t si = 0;
    for (uint32_t i = 1; i < segs.count; i++)
        if (blockIdx.x >= segs.cb0[i]) si = i;
    const uint32_t c0 = (blockIdx.x - segs.cb0[si]) * COLS;
    const uint32_t m = segs.m[si], lp = segs.lines_p[si];
    const int32_t* __restrict__ part = segs.part[si];
    const uint32_t ck = (ax.op >> 8) & 3;
    const bool pb = (ax.op & ro::F_P_BCAST) != 0;
    // element e of the tile: row e / COLS, column c0 + e % COLS
    auto epi_in = [&](uint32_t e) {
        SkinnyEpiIn in;
        const uint32_t row = e / COLS, col = c0 + e % COLS;
        if (row >= n || col >= m) return in;
#pragma unroll
        for (uint32_t sl = 0; sl < kSpSlabs; sl++)
            if (sl < nslab) in.cs[sl] = (uint32_t)part[(uint64_t)sl * lp + col];
        if constexpr (XK != 0) {
            in.prm = *reinterpret_cast<const uint4*>(ax.params + 16u * (pb ? 0u : col));
            const uint64_t ex = (uint64_t)row * m + col;
            if constexpr (XK == 1) in.x = reinterpret_cast<const int16_t*>(ax.x)[ex];
            else in.x = reinterpret_cast<const int32_t*>(ax.x)[ex];
        }
        return in;
    };
    constexpr uint32_t PRE = sp_pre(NB);
    SkinnyEpiIn pre[PRE];
#pragma unroll
    for (uint32_t i = 0; i < PRE; i++) pre[i] = epi_in(threadIdx.x + i * blockDim.x);
    const int8_t* bh[NB];
    const int8_t* bl[NB];
#pragma unroll
    for (uint32_t b = 0; b < NB; b++) {
        bh[b] = segs.hi[si] + (uint64_t)(c0 + 16 * b) * kp;
        bl[b] = segs.lo[si] + (uint64_t)(c0 + 16 * b) * kp;
    }
    skinny_products<NB, SAT>(a, n, k, kp, bh, bl, red, rsum);
    int16_t* __restrict__ c = segs.c[si];
    auto store = [&](uint32_t e, const SkinnyEpiIn& in) {
        const uint32_t row = e / COLS, cl = e - row * COLS, col = c0 + cl;
        if (row >= n || col >= m) return;
        const uint32_t cs = skinny_colsum(in.cs, part, nslab, lp, col);
        const int16_t y = SAT ? skinny_value_sat(red, rsum, W, COLS, row, cl, k, cs)
                              : skinny_value(red, rsum, W, COLS, row, cl, k, cs);
        const uint64_t eo = (uint64_t)row * m + col;
        c[eo] = y;
        if constexpr (XK != 0) {
            const ro::i64 o = ro::copy_addx(in.x, y, ro::param_of(in.prm), ax.op, ax.bq_sh, ck);
            if (ck == 0) reinterpret_cast<int16_t*>(ax.out)[eo] = (int16_t)o;
            else reinterpret_cast<int32_t*>(ax.out)[eo] = (int32_t)o;
        }
    };
#pragma unroll
    for (uint32_t i = 0; i < PRE; i++)
        if (threadIdx.x + i * blockDim.x < 16 * COLS) store(threadIdx.x + i * blockDim.x, pre[i]);
    for (uint32_t e = threadIdx.x + PRE * blockDim.x; e < 16 * COLS; e += blockDim.x) store(e, epi_in(e));
}

// The MULACT job over a gate and an up product of the same A (segments 0 and 1, m columns
// each): a workgroup's NB blocks are NB / 2 blocks of gate columns and the same columns of up,
// and its stores write both products and out = MULACT(gate, up) with the job's parameters.
struct SkinnyMulact {
    int16_t* out;
    const uint8_t* params;
    uint32_t bcast;
    const uint8_t* tab;       // the row-ops table image (the sigmoid)
};

struct SkinnyPairIn {
    uint32_t cg[kSpSlabs] = {0, 0, 0, 0}, cu[kSpSlabs] = {0, 0, 0, 0};
    uint4 prm{};
};

template <uint32_t NB>
__global__ __launch_bounds__(64 * sp_max_waves(NB)) void skinny_mulact_kernel(const int16_t* __restrict__ a, uint32_t n,
                                                                        uint32_t k, uint32_t kp, uint32_t nslab,
                                                                        SkinnyPlaneSegs segs, SkinnyMulact mj) {
    constexpr uint32_t COLS = 16 * NB, H = COLS / 2;
    extern __shared__ __attribute__((aligned(16))) uint32_t sp_lds[];
    const uint32_t W = blockDim.x >> 6;
    uint32_t* red = sp_lds;
    int32_t* rsum = reinterpret_cast<int32_t*>(sp_lds + W * 16 * COLS);
    const uint32_t c0 = blockIdx.x * H, m = segs.m[0], lp = segs.lines_p[0];
    auto epi_in = [&](uint32_t e) {
        SkinnyPairIn in;
        const uint32_t row = e / H, col = c0 + e % H;
        if (row >= n || col >= m) return in;
#pragma unroll
        for (uint32_t sl = 0; sl < kSpSlabs; sl++)
            if (sl < nslab) {
                in.cg[sl] = (uint32_t)segs.part[0][(uint64_t)sl * lp + col];
                in.cu[sl] = (uint32_t)segs.part[1][(uint64_t)sl * segs.lines_p[1] + col];
            }
        in.prm = *reinterpret_cast<const uint4*>(mj.params + 16u * (mj.bcast ? 0u : col));
        return in;
    };
    const SkinnyPairIn pre = epi_in(threadIdx.x);
    const int8_t* bh[NB];
    const int8_t* bl[NB];
#pragma unroll
    for (uint32_t b = 0; b < NB; b++) {
        const uint32_t sg = b < NB / 2 ? 0u : 1u, cb = c0 + 16 * (b % (NB / 2));
        bh[b] = segs.hi[sg] + (uint64_t)cb * kp;
        bl[b] = segs.lo[sg] + (uint64_t)cb * kp;
    }
    skinny_products<NB>(a, n, k, kp, bh, bl, red, rsum);
    auto store = [&](uint32_t e, const SkinnyPairIn& in) {
        const uint32_t row = e / H, cl = e - row * H, col = c0 + cl;
        if (row >= n || col >= m) return;
        const int16_t gv = skinny_value(red, rsum, W, COLS, row, cl, k, skinny_colsum(in.cg, segs.part[0], nslab, lp, col));
        const int16_t uv = skinny_value(red, rsum, W, COLS, row, H + cl, k,
                                        skinny_colsum(in.cu, segs.part[1], nslab, segs.lines_p[1], col));
        const uint64_t eo = (uint64_t)row * m + col;
        segs.c[0][eo] = gv;
        segs.c[1][eo] = uv;
        mj.out[eo] = (int16_t)ro::mulact_elem(gv, uv, ro::param_of(in.prm), mj.tab);
    };
    if (threadIdx.x < 16 * H) store(threadIdx.x, pre);
    for (uint32_t e = threadIdx.x + blockDim.x; e < 16 * H; e += blockDim.x) store(e, epi_in(e));
}

// ---------------------------------------------------------------- drivers
// The tile of a product: kernel variant, rows, columns and workgroups a compute unit holds.
struct GemmPlan {
    uint32_t id, tm, tn, per_cu;
};
constexpr GemmPlan kPlan128{0, 128, 128, 2}, kPlan256{1, 256, 128, 1};   // gemm_planes_kernel
constexpr GemmPlan kRing64{2, 64, 64, 2}, kRing128{3, 128, 128, 1};      // gemm_ring_kernel

// Byte planes [slices][lines_p][kp] of one operand and its partial line sums
// [slices][nslab][lines_p].
struct Planes {
    int8_t *hi, *lo;
    int32_t* part;
    uint32_t lines_p, kp, nslab, slices;
    GemmPlan plan = kPlan128;            // the GEMM's tile when this is the A operand
    uint32_t rows = 0;                   // real lines (the rest up to lines_p are padding)
    uint32_t sums = 0;                   // partial line sums per line (0: one per slab)
    uint32_t nsum() const { return sums ? sums : nslab; }
    size_t bytes() const {
        return (size_t)slices * lines_p * kp * 2 + (size_t)slices * nslab * lines_p * 4 + 1024;
    }
    void carve(char*& p) {
        hi = reinterpret_cast<int8_t*>(p); p += (size_t)slices * lines_p * kp;
        lo = reinterpret_cast<int8_t*>(p); p += (size_t)slices * lines_p * kp;
        part = reinterpret_cast<int32_t*>(p); p += (size_t)slices * nslab * lines_p * 4;
        p = reinterpret_cast<char*>(round_up(reinterpret_cast<uintptr_t>(p), 256));
    }
};

template <class Src, bool KFast>
int run_split(const Src& src, uint64_t src_slice, Planes& pl, hipStream_t s) {
    CM_LAUNCH("split_kernel", (split_kernel<Src, KFast>), dim3(pl.lines_p / 64, pl.nslab, pl.slices), dim3(256),
                       0, s, src, src_slice, pl.hi, pl.lo, pl.part, pl.lines_p, pl.kp, pl.nslab);
    return CM_OK;
}

// k slices of a wrap-mode product of `tiles` tiles of a plan: as many as fill the workgroup slots
// once, each of at least 12 k steps of a 64 x 64 tile or 8 of a larger one (a slice's partials cost a
// round trip to the coherence point: 128 x 3072 x 768 on 64 x 64 tiles takes 11.9 us in 2 slices, 9.7 in 4
// of 12 steps, 10.6 in 8; 1280 x 1536 x 2048 on 128 x 128 tiles 31.9 unsplit, 30.7 in 3 of 8).
uint32_t gemm_slices(const GemmPlan& pl, uint64_t tiles, uint32_t nk, uint32_t cus) {
    return (uint32_t)std::min<uint64_t>((uint64_t)cus * pl.per_cu / tiles, nk / (pl.tm == 64 ? 12 : 8));
}

// The tile of an n x m output of `batch` slices and nk k steps, where a product by the int32-wrap
// rule (`wrap`) may be split over k; measured (us, k = 768 unless given):
//   - 64 x 64 tiles on the four-stage ring while they fit the slots once (two workgroups a unit):
//     128 x 2304 6.9 (128 x 128 tiles, two stages: 13.2), 1040 x 768 7.7 (15.2), 512 x 3072 10.0
//     (13.6); and for outputs of at most 64 rows at any width: 24 x 100352 of k 192 18.9 (64 x 128
//     tiles, two stages: 23.6);
//   - but 128 x 128 tiles, split over k, for a wrap product whose 64 x 64 tiles would take at most 2 slices
//     of 48 steps or more: they read half the bytes a product (in 3 slices or more the 64 x 64 tiles stay
//     ahead: 384 x 1024 of k 16384 45.3 in 5, 57.1; so do they below 96 steps where the larger tiles pad
//     more than an eighth: 3606 x 317 of k 11696 takes 112 on those, 145 on 64 x 64; and below 64 where two
//     slices fill less than 7 of 8 units: an encoder layer of 12 x 176 tokens, 2112 x 768 of k 3072 in it,
//     162.2 on 64 x 64, 164.8).  On the ring, one workgroup a unit (A's planes given): 2000 x 1000 of k
//     3072 33.6 in 2 (64 x 64 34.5; two stages, in 4, 38.8), 1250 x 1000 of k 4096 31.2 in 3 (36.2; in 6,
//     37.4), 640 x 2048 of k 8192 56.1 in 3 (77.0; in 6, 56.5).  On the two stages, two workgroups a unit,
//     where they fill the units better or a slice of the ring is long, from 64 steps over whole tiles (1536
//     x 1024 of k 4096 35.9 in 5, the ring in 2 36.5; 2048 x 1024 of k 16384 143.5 in 4, 151.2), from 80
//     over ragged ones, whose stores cost them more (1500 x 1024 of k 4096 39.0 and 37.0, of k 6144 50.1
//     and 50.6);
//   - 128 x 128 tiles on the ring with 8 waves while they fit one to a unit: 1040 x 2304 15.1 (two
//     stages 16.7), 576 x 6272 of k 128 8.0 (11.8), 3072 x 768 14.4 (14.3); but a wrap product that
//     splits in 3 or more keeps the two-stage kernel, two workgroups a unit: 3072 x 768 of k 3072
//     45.0 (ring unsplit 52.6), while 3072 x 1024 of k 4096 takes 68.3 on the ring, 70.1 split in 2; in 2
//     slices of 48 steps or more where they fill 3 of 4 slots: 2048 x 2048 of k 8192 129.2 (142.4), of k 4096
//     73.2 (72.7), 1536 x 2048 of k 8192 118.2 (119.1);
//   - above, 256 x 128 tiles (one workgroup of 8 waves a unit, three stages) where their rounds
//     over the units cost no more than the 128 x 128 tiles' (a round of them takes 22 - 25, of 128
//     x 128 tiles 12.6 per tile a unit): 3072 x 2304 24.7 (26.7), 3072 x 3072 44.2 (37.8); of 8 steps or
//     fewer, where a workgroup alone on its unit pays its start and its stores in full, only a single round
//     without a padded half tile: 1024 x 8192 of k 512 26.2 (26.8), 640 x 8192 of k 512 26.3 (24.2), 4096 x 6000 of
//     k 256 50.4 (45.0).
GemmPlan gemm_plan(uint32_t n, uint32_t m, uint32_t batch, uint32_t nk, bool wrap, uint32_t cus) {
    auto tiles = [&](const GemmPlan& pl) { return (uint64_t)ceil_div(n, pl.tm) * ceil_div(m, pl.tn) * batch; };
    auto slices = [&](const GemmPlan& pl) { return std::max(1u, gemm_slices(pl, tiles(pl), nk, cus)); };
    const uint64_t t128 = tiles(kPlan128), t256 = tiles(kPlan256);
    if (n <= 64 || tiles(kRing64) <= 2ull * cus) {
        const uint32_t few = slices(kRing64), ring = slices(kRing128), two = slices(kPlan128);
        if (n <= 64 || !wrap || few > 2 || nk / few < 48) return kRing64;
        if (nk / few < 96 && (ring < 2 || 32 * t128 > 9 * tiles(kRing64))) return kRing64;
        if (nk / few < 64 && ring == 2 && 8 * t128 < 7 * (cus / 2)) return kRing64;
        const uint32_t steps = n % 128 == 0 && m % 128 == 0 ? 64 : 80;
        return nk >= steps && (nk / ring >= steps || 2 * ring < two) ? kPlan128 : kRing128;
    }
    if (t128 <= cus) {
        const uint32_t two = slices(kPlan128);
        return wrap && (two >= 3 || (two == 2 && nk >= 96 && 4 * t128 >= 3ull * cus)) ? kPlan128 : kRing128;
    }
    if (2 * ((t256 + cus - 1) / cus) > (t128 + cus - 1) / cus) return kPlan128;
    return nk > 8 || (t256 <= cus && 2 * t256 == t128) ? kPlan256 : kPlan128;
}

// Tile columns of the strips tile_pos walks: the square root of an XCD's share of the tiles.
uint32_t gemm_strip(uint32_t tiles, uint32_t tiles_c) {
    uint32_t w = 1;
    while ((w + 1) * (w + 1) * 8 <= tiles) w++;
    return std::min(w, tiles_c);
}

template <class Epi>
int run_gemm(const Planes& A, const Planes& B, uint32_t batch, uint32_t k, Epi epi, hipStream_t s,
             int32_t* pout = nullptr, uint32_t ksteps = 0, uint32_t* tcnt = nullptr) {
    const GemmPlan pl = A.plan;
    const uint32_t tiles_r = ceil_div(A.rows, pl.tm), tiles_c = ceil_div(B.rows, pl.tn);
    if ((uint64_t)tiles_r * pl.tm > A.lines_p || (uint64_t)tiles_c * pl.tn > B.lines_p)
        return fail(CM_EINVAL, "gemm: %u x %u tiles past %u x %u plane lines", tiles_r, tiles_c, A.lines_p, B.lines_p);
    const uint64_t a_slice = A.slices > 1 ? (uint64_t)A.lines_p * A.kp : 0;
    const uint64_t b_slice = B.slices > 1 ? (uint64_t)B.lines_p * B.kp : 0;
    const uint64_t rp_slice = A.slices > 1 ? (uint64_t)A.nslab * A.lines_p : 0;
    const uint64_t cp_slice = B.slices > 1 ? (uint64_t)B.nslab * B.lines_p : 0;
    if (ksteps && tcnt == nullptr) return fail(CM_EINVAL, "gemm: a split over k needs the arrival counts");
    const uint32_t mode = ksteps ? kSplitFix : (epi.wrap ? kWrap : (k <= 8192 ? kSatNarrow : kSatWide));
    const uint32_t nz = ksteps ? ceil_div(A.kp / BK, ksteps) : 1;
    const uint32_t xw = gemm_strip(tiles_r * tiles_c, tiles_c);
    const dim3 grid(tiles_r * tiles_c, batch, nz);
#define CM_GEMM(NT, ...)                                                                                             \
    CM_LAUNCH("gemm_planes_kernel", (__VA_ARGS__), grid, dim3(NT), 0, s, A.hi, A.lo, A.part, a_slice, rp_slice,       \
              A.lines_p, B.hi, B.lo, B.part, b_slice, cp_slice, B.lines_p, B.nslab, A.nsum(), tiles_r, tiles_c, xw,   \
              A.kp, (int32_t)(64 * k), mode, pout, ksteps, tcnt, epi)
    switch (pl.id) {
    case kPlan256.id: CM_GEMM(512, gemm_planes_kernel<4, 3, Epi>); break;
    case kRing64.id: CM_GEMM(256, gemm_ring_kernel<1, 1, 2, 2, Epi>); break;
    case kRing128.id: CM_GEMM(512, gemm_ring_kernel<1, 2, 4, 2, Epi>); break;
    default: CM_GEMM(256, gemm_planes_kernel<2, 2, Epi>); break;
    }
#undef CM_GEMM
    return CM_OK;
}

// k steps per slice of a wrap-mode product (0: no split).
uint32_t gemm_ksteps(const GemmPlan& pl, uint32_t tiles, uint32_t kp, const DeviceState* st) {
    const uint32_t nk = kp / BK, nz = gemm_slices(pl, tiles, nk, st->cus);
    return nz < 2 ? 0 : ceil_div(nk, nz);
}

Planes make_planes(uint32_t lines, uint32_t kp, uint32_t slices, uint32_t align = 128) {
    Planes p{};
    p.lines_p = (uint32_t)round_up(lines, align);
    p.rows = lines;
    p.kp = kp;
    p.nslab = ceil_div(kp, SLAB);
    p.slices = slices;
    return p;
}

// A's planes for a product by `plan`.
Planes make_a_planes(uint32_t lines, uint32_t kp, uint32_t slices, const GemmPlan& plan) {
    Planes p = make_planes(lines, kp, slices, plan.tm);
    p.plan = plan;
    return p;
}

}  // namespace
}  // namespace cm

namespace cm {
namespace {

int matmul_check(uint32_t k, uint32_t gemv_kw, int64_t a_bs, int64_t b_bs, int64_t c_bs, uint32_t b_packed = 0) {
    // the limb sums HL + LH stay exact in int32 for k <= 32768
    if (k == 0 || k > 32768) return fail(CM_EINVAL, "matmul: k = %u outside 1 .. 32768", k);
    if (gemv_kw && gemv_kw != 1 && gemv_kw != 2 && gemv_kw != 4 && gemv_kw != 8)
        return fail(CM_EINVAL, "matmul: gemv_kw %u", gemv_kw);
    if (gemv_kw > 1 && (k % (16 * gemv_kw)))
        return fail(CM_EINVAL, "matmul: k %u not a multiple of 16 * gemv_kw", k);
    if (b_packed > 2 || (b_packed && gemv_kw)) return fail(CM_EINVAL, "matmul: b_packed %u with gemv_kw %u", b_packed, gemv_kw);
    if (a_bs < 0 || b_bs < 0 || c_bs < 0) return fail(CM_EINVAL, "matmul: negative batch stride");
    return CM_OK;
}

// Planes of rows with k contiguous (lda elements apart): the short-row kernel for kp <= 256, else a wavefront per row and slab.
int split_row_lines(const int16_t* a, Slices a_slice, uint64_t lda, uint32_t n, uint32_t k, Planes& P,
                    hipStream_t s) {
    if (P.kp <= 256) {
#define CM_SHORT(G)                                                                                            \
    CM_LAUNCH("split_rows_kernel", split_rows_short_kernel<G>, dim3(ceil_div(P.lines_p, 4 * (64 / G)), 1, P.slices), \
              dim3(256), 0, s, a, a_slice, lda, n, k, P.hi, P.lo, P.part, P.lines_p, P.kp)
        if (P.kp == 64) { CM_SHORT(8); } else if (P.kp == 128) { CM_SHORT(16); } else { CM_SHORT(32); }
#undef CM_SHORT
        return CM_OK;
    }
    CM_LAUNCH("split_rows_kernel", split_rows_kernel, dim3(P.lines_p / 4, P.nslab, P.slices), dim3(256), 0, s, a,
              a_slice, lda, n, k, P.hi, P.lo, P.part, P.lines_p, P.kp, P.nslab);
    return CM_OK;
}

// A's planes: row-major [n][k] slices at a_slice elements (0: one slice).
int split_a(const int16_t* a, uint64_t a_slice, uint32_t n, uint32_t k, Planes& A, hipStream_t s) {
    return split_row_lines(a, Slices{a_slice}, k, n, k, A, s);
}

// B's planes from its image (row-major, packed 32-column tiles or the GEMV image).
int split_b(const int16_t* b, uint64_t b_slice, uint32_t k, uint32_t m, uint32_t b_packed, uint32_t gemv_kw,
            Planes& B, hipStream_t s) {
    const uint32_t layout = gemv_kw ? 2 : (b_packed == 2 ? 3 : (b_packed ? 1 : 0));
    if (layout == 3)
        return split_row_lines(b, Slices{b_slice}, k, m, k, B, s);    // B's lines are rows with k contiguous
    if (layout <= 1 || (layout == 2 && gemv_kw == 1)) {
        CM_LAUNCH("split_cols_kernel", split_cols_kernel, dim3(B.lines_p / 32, B.nslab, B.slices), dim3(256), 0, s,
                  b, Slices{b_slice}, (uint64_t)m, layout == 1 ? 1u : 0u, m, k, B.hi, B.lo, B.part, B.lines_p, B.kp,
                  B.nslab);
        return CM_OK;
    }
    return run_split<SrcGemvB, false>(SrcGemvB{b, k, m, gemv_kw}, b_slice, B, s);
}

// The skinny path of cm_matmul (wrap32, n <= 32): slices of kSkinnyKc k.
// Skinny products of the same A (n rows, k) into `count` segments, or one product over
// `batch` slices (count 1); the partials of all segments in one workspace, one reduce launch.
int skinny_run(const int16_t* a, uint32_t n, uint32_t k, uint32_t batch, int64_t a_bs, int64_t b_bs, int64_t c_bs,
               uint32_t count, const int16_t* const* b, int16_t* const* c, const uint32_t* m, uint32_t b_packed,
               DeviceState* st, hipStream_t s, const WsRegion* fixed = nullptr) {
    const uint32_t nks = ceil_div(k, kSkinnyKc);
    SkinnySegs segs{};
    segs.count = count;
    uint32_t cbs = 0;
    uint64_t pairs = 0;
    size_t pbytes = 0;
    for (uint32_t i = 0; i < count; i++) {
        segs.b[i] = b[i];
        segs.c[i] = c[i];
        segs.m[i] = m[i];
        segs.cb0[i] = cbs;
        segs.pair0[i] = pairs;
        cbs += ceil_div(m[i], 128);
        pairs += (uint64_t)batch * n * m[i] / 2;
        pbytes += (size_t)batch * nks * n * m[i] * 4;
    }
    if (nks > 65535 || batch > 65535) return fail(CM_EINVAL, "matmul: skinny grid %u x %u x %u", cbs, nks, batch);
    if (nks > 1) {
        void* ws;
        int rc = take_workspace(st, fixed, pbytes, &ws, s);
        if (rc) return rc;
        int32_t* p = static_cast<int32_t*>(ws);
        for (uint32_t i = 0; i < count; i++) {
            segs.part[i] = p;
            p += (size_t)batch * nks * n * m[i];
        }
    }
    const dim3 grid(cbs, nks, batch);
#define CM_SKINNY(NR, BL)                                                                                         \
    CM_LAUNCH("skinny_wrap_kernel", (skinny_wrap_kernel<NR, BL>), grid, dim3(64), 0, s, a, (uint64_t)a_bs, segs,   \
              (uint64_t)b_bs, (uint64_t)c_bs, n, k)
#define CM_SKINNY_BL(NR) \
    if (b_packed == 2) { CM_SKINNY(NR, 2); } else if (b_packed) { CM_SKINNY(NR, 1); } else { CM_SKINNY(NR, 0); }
    if (n <= 8) { CM_SKINNY_BL(8) } else if (n <= 16) { CM_SKINNY_BL(16) } else { CM_SKINNY_BL(32) }
#undef CM_SKINNY_BL
#undef CM_SKINNY
    if (nks > 1) {
        const unsigned blocks = (unsigned)std::min<uint64_t>((pairs + 255) / 256, (uint64_t)st->cus * 8);
        CM_LAUNCH("skinny_reduce_kernel", skinny_reduce_kernel, dim3(blocks), dim3(256), 0, s, segs, (uint64_t)c_bs,
                  n, nks, batch, pairs);
    }
    return CM_OK;
}

int skinny_wrap(const int16_t* a, const int16_t* b, int16_t* c, uint32_t n, uint32_t k, uint32_t m, uint32_t batch,
                int64_t a_bs, int64_t b_bs, int64_t c_bs, uint32_t b_packed, DeviceState* st, hipStream_t s,
                const WsRegion* fixed) {
    return skinny_run(a, n, k, batch, a_bs, b_bs, c_bs, 1, &b, &c, &m, b_packed, st, s, fixed);
}

// The wrap-mode split over k for a matmul of this shape: k steps per slice (0: none) and the
// bytes of its int32 partials.
uint32_t matmul_ksteps(const Planes& A, const Planes& B, uint32_t n, uint32_t m, uint32_t batch, uint32_t wrap32,
                       const DeviceState* st, size_t* bytes) {
    const uint32_t tiles = ceil_div(n, A.plan.tm) * ceil_div(m, A.plan.tn) * batch;
    const uint32_t ks = wrap32 ? gemm_ksteps(A.plan, tiles, A.kp, st) : 0;
    // the partials of every slice, whole tiles (split_fixup's layout)
    *bytes = ks ? (size_t)ceil_div(A.kp / BK, ks) * tiles * A.plan.tm * A.plan.tn * 4 : 0;
    return ks;
}

int gemm_out(const Planes& A, const Planes& B, int16_t* c, uint32_t n, uint32_t k, uint32_t m, uint32_t batch,
             int64_t c_bs, uint32_t wrap32, hipStream_t s, const DeviceState* st, int32_t* pout = nullptr,
             uint32_t ksteps = 0) {
    const bool pairs = (reinterpret_cast<uintptr_t>(c) & 3) == 0 && (m & 1) == 0 && (c_bs & 1) == 0;
    EpiMatmul epi{c, (uint64_t)c_bs, n, m, wrap32 ? 1u : 0u, pairs ? 1u : 0u};
    // a split product is finished by the last slice of each tile (one launch): an arrival
    // count per tile (a split has at most one tile per compute unit, gemm_ksteps)
    const uint64_t tiles = (uint64_t)ceil_div(A.rows, A.plan.tm) * ceil_div(m, A.plan.tn) * batch;
    if (ksteps && tiles > st->split_cnt_n)
        return fail(CM_EINVAL, "gemm: %llu split tiles past the %u arrival counts", (unsigned long long)tiles,
                    st->split_cnt_n);
    return run_gemm(A, B, batch, k, epi, s, pout, ksteps, ksteps ? st->split_cnt : nullptr);
}

}  // namespace
}  // namespace cm

namespace cm {
namespace {

// cm_matmul with its workspace from `fixed` (nullptr: the grow-only workspace).
int matmul_run(const int16_t* a, const int16_t* b, int16_t* c, uint32_t n, uint32_t k, uint32_t m, uint32_t batch,
               int64_t a_bs, int64_t b_bs, int64_t c_bs, uint32_t b_packed, uint32_t gemv_kw, uint32_t wrap32,
               hipStream_t s, DeviceState* st, const WsRegion* fixed) {
    if (n == 0 || m == 0 || batch == 0) return CM_OK;
    int rc = matmul_check(k, gemv_kw, a_bs, b_bs, c_bs, b_packed);
    if (rc) return rc;
    if (wrap32 && n <= 32 && gemv_kw == 0 && (m & 1) == 0 && (k & 1) == 0 && (reinterpret_cast<uintptr_t>(a) & 3) == 0 &&
        (reinterpret_cast<uintptr_t>(b) & 3) == 0 && (reinterpret_cast<uintptr_t>(c) & 3) == 0 && (a_bs & 1) == 0 &&
        (b_bs & 1) == 0 && (c_bs & 1) == 0 && (b_packed != 1 || (m & 31) == 0) &&
        (b_packed != 2 || ((k & 7) == 0 && aligned16(b) && (b_bs & 7) == 0)))
        return skinny_wrap(a, b, c, n, k, m, batch, a_bs, b_bs, c_bs, b_packed, st, s, fixed);
    const uint32_t kp = (uint32_t)round_up(k, BK);
    const uint32_t sa = (batch > 1 && a_bs != 0) ? batch : 1, sb = (batch > 1 && b_bs != 0) ? batch : 1;
    Planes A = make_a_planes(n, kp, sa, gemm_plan(n, m, batch, kp / BK, wrap32, st->cus)), B = make_planes(m, kp, sb);
    size_t pbytes;
    uint32_t ksteps = matmul_ksteps(A, B, n, m, batch, wrap32, st, &pbytes);
    if (fixed != nullptr && A.bytes() + B.bytes() + pbytes > fixed->cap) {
        // the least a product needs: rows rounded up to 64, no partials
        A = make_a_planes(n, kp, sa, kRing64);
        ksteps = 0;
        pbytes = 0;
    }
    void* ws;
    rc = take_workspace(st, fixed, A.bytes() + B.bytes() + pbytes, &ws, s);
    if (rc) return rc;
    char* p = static_cast<char*>(ws);
    A.carve(p);
    B.carve(p);
    const uint64_t a_slice = sa > 1 ? (uint64_t)a_bs : 0, b_slice = sb > 1 ? (uint64_t)b_bs : 0;
    rc = split_a(a, a_slice, n, k, A, s);
    if (rc) return rc;
    rc = split_b(b, b_slice, k, m, b_packed, gemv_kw, B, s);
    if (rc) return rc;
    return gemm_out(A, B, c, n, k, m, batch, c_bs, wrap32, s, st, reinterpret_cast<int32_t*>(p), ksteps);
}

// The no-allocation scratch: every call of cm_matmul_noalloc on a device takes its planes, line
// sums and split-k partials from that device's copy of this array (the code object holds one
// per device from load to process end).  Host code never passes `scratch` itself: its
// device address per device comes from hipGetSymbolAddress at set-up (DeviceState::scratch).
constexpr size_t kScratchBytes = CM_NOALLOC_MAX_BYTES;
static __device__ __align__(256) uint8_t scratch[kScratchBytes];

// The arrival counts of the split-k products finished in place (kSplitFix), one per output
// tile and batch slice of a launch: zero from load, and every launch leaves them zero (the
// last slice of a tile resets its count), so they need no clearing between launches or graph
// replays.  Launches that overlap on one device (other streams) must not both split.
constexpr uint32_t kSplitCounts = 16384;
static __device__ __align__(256) uint32_t split_counts[kSplitCounts];

}  // namespace

int gemm_scratch_setup(DeviceState* st) {
    void* ptr = nullptr;
    CM_HIP_CHECK(hipGetSymbolAddress((void**)&ptr, HIP_SYMBOL(scratch)));
    if (ptr == nullptr || (reinterpret_cast<uintptr_t>(ptr) & 255))
        return fail(CM_EHIP, "no-allocation scratch: unusable device address %p", ptr);
    st->scratch = ptr;
    st->scratch_bytes = kScratchBytes;
    void* cp = nullptr;
    CM_HIP_CHECK(hipGetSymbolAddress(&cp, HIP_SYMBOL(split_counts)));
    if (cp == nullptr) return fail(CM_EHIP, "split-k arrival counts: no device address");
    st->split_cnt = static_cast<uint32_t*>(cp);
    st->split_cnt_n = kSplitCounts;
    return CM_OK;
}

}  // namespace cm

extern "C" int cm_matmul(const int16_t* a, const int16_t* b, int16_t* c, uint32_t n, uint32_t k,
                         uint32_t m, uint32_t batch, int64_t a_bs, int64_t b_bs, int64_t c_bs,
                         uint32_t b_packed, uint32_t gemv_kw, uint32_t wrap32, void* stream) {
    using namespace cm;
    DeviceState* st;
    int rc = state(&st);
    if (rc) return rc;
    return matmul_run(a, b, c, n, k, m, batch, a_bs, b_bs, c_bs, b_packed, gemv_kw, wrap32, as_stream(stream), st,
                      nullptr);
}

extern "C" int cm_matmul_noalloc(const int16_t* a, const int16_t* b, int16_t* c, uint32_t n, uint32_t k,
                                 uint32_t m, uint32_t batch, int64_t a_bs, int64_t b_bs, int64_t c_bs,
                                 uint32_t b_packed, uint32_t gemv_kw, uint32_t wrap32, void* stream) {
    using namespace cm;
    DeviceState* st;
    int rc = state_ready(&st);                       // no set-up here: that allocates the unit tables
    if (rc) return rc;
    if (st->scratch == nullptr) return fail(CM_EINVAL, "no-allocation scratch not set up on this device");
    const WsRegion region{st->scratch, st->scratch_bytes};
    return matmul_run(a, b, c, n, k, m, batch, a_bs, b_bs, c_bs, b_packed, gemv_kw, wrap32, as_stream(stream), st,
                      &region);
}

extern "C" size_t cm_matmul_b_planes_bytes(uint32_t k, uint32_t m, uint32_t b_slices) {
    using namespace cm;
    if (k == 0 || m == 0 || b_slices == 0) return 0;
    return make_planes(m, (uint32_t)round_up(k, BK), b_slices).bytes();
}

extern "C" int cm_matmul_split_b(const int16_t* b, void* planes, uint32_t k, uint32_t m, uint32_t b_slices,
                                 int64_t b_bs, uint32_t b_packed, uint32_t gemv_kw, void* stream) {
    using namespace cm;
    DeviceState* st;
    int rc = state(&st);
    if (rc) return rc;
    if (m == 0 || b_slices == 0) return CM_OK;
    rc = matmul_check(k, gemv_kw, 0, b_bs, 0, b_packed);
    if (rc) return rc;
    if (reinterpret_cast<uintptr_t>(planes) & 255) return fail(CM_EALIGN, "matmul: b planes not 256-byte aligned");
    Planes B = make_planes(m, (uint32_t)round_up(k, BK), b_slices);
    char* p = static_cast<char*>(planes);
    B.carve(p);
    return split_b(b, b_slices > 1 ? (uint64_t)b_bs : 0, k, m, b_packed, gemv_kw, B, as_stream(stream));
}

extern "C" int cm_matmul_planes(const int16_t* a, const void* b_planes, int16_t* c, uint32_t n, uint32_t k,
                                uint32_t m, uint32_t batch, int64_t a_bs, uint32_t b_slices, int64_t c_bs,
                                uint32_t wrap32, void* stream) {
    using namespace cm;
    DeviceState* st;
    int rc = state(&st);
    if (rc) return rc;
    if (n == 0 || m == 0 || batch == 0) return CM_OK;
    rc = matmul_check(k, 0, a_bs, 0, c_bs);
    if (rc) return rc;
    if (b_slices != 1 && b_slices != batch) return fail(CM_EINVAL, "matmul: %u b slices for batch %u", b_slices, batch);
    if (reinterpret_cast<uintptr_t>(b_planes) & 255) return fail(CM_EALIGN, "matmul: b planes not 256-byte aligned");
    hipStream_t s = as_stream(stream);
    const uint32_t kp = (uint32_t)round_up(k, BK);
    const uint32_t sa = (batch > 1 && a_bs != 0) ? batch : 1;
    Planes A = make_a_planes(n, kp, sa, gemm_plan(n, m, batch, kp / BK, wrap32, st->cus)), B = make_planes(m, kp, b_slices);
    size_t pbytes;
    const uint32_t ksteps = matmul_ksteps(A, B, n, m, batch, wrap32, st, &pbytes);
    void* ws;
    rc = workspace(st, A.bytes() + pbytes, &ws, s);
    if (rc) return rc;
    char* p = static_cast<char*>(ws);
    A.carve(p);
    char* q = static_cast<char*>(const_cast<void*>(b_planes));
    B.carve(q);
    rc = split_a(a, sa > 1 ? (uint64_t)a_bs : 0, n, k, A, s);
    if (rc) return rc;
    return gemm_out(A, B, c, n, k, m, batch, c_bs, wrap32, s, st, reinterpret_cast<int32_t*>(p), ksteps);
}

extern "C" size_t cm_matmul_a_planes_bytes(uint32_t n, uint32_t k, uint32_t nsum) {
    return cm::a_planes_bytes(n, k, nsum);
}

extern "C" int cm_matmul_aplanes(const void* a_planes, uint32_t nsum, const void* b_planes, int16_t* c, uint32_t n,
                                 uint32_t k, uint32_t m, uint32_t wrap32, void* stream) {
    using namespace cm;
    DeviceState* st;
    int rc = state(&st);
    if (rc) return rc;
    if (n == 0 || m == 0) return CM_OK;
    rc = matmul_check(k, 0, 0, 0, 0);
    if (rc) return rc;
    if ((k % BK) || nsum == 0 || nsum > 64) return fail(CM_EINVAL, "matmul: A planes of k %u (a multiple of 64), %u sums", k, nsum);
    if ((reinterpret_cast<uintptr_t>(a_planes) & 255) || (reinterpret_cast<uintptr_t>(b_planes) & 255))
        return fail(CM_EALIGN, "matmul: planes not 256-byte aligned");
    hipStream_t s = as_stream(stream);
    const APlanes ap = a_planes_view(const_cast<void*>(a_planes), n, k, nsum);
    Planes A = make_a_planes(n, k, 1, gemm_plan(n, m, 1, k / BK, wrap32, st->cus)), B = make_planes(m, k, 1);
    A.hi = ap.hi;
    A.lo = ap.lo;
    A.part = ap.part;
    A.lines_p = ap.lines;
    A.sums = nsum;
    char* q = static_cast<char*>(const_cast<void*>(b_planes));
    B.carve(q);
    size_t pbytes;
    const uint32_t ksteps = matmul_ksteps(A, B, n, m, 1, wrap32, st, &pbytes);
    void* ws = nullptr;
    if (pbytes) {
        rc = workspace(st, pbytes, &ws, s);
        if (rc) return rc;
    }
    return gemm_out(A, B, c, n, k, m, 1, 0, wrap32, s, st, static_cast<int32_t*>(ws), ksteps);
}

namespace cm {
namespace {

struct ConvGeom {
    uint32_t batch, in_ch, in_h, in_w, out_ch, out_h, out_w, kh, kw, sh, sw, dh, dw, pt, pl;
    uint32_t cs, cn, gs, wrap;          // the y pattern (cs = plane without one), int32 wrap
    uint32_t plane() const { return out_h * out_w; }
    // 1x1 stride-1 unpadded, same plane in and out
    bool pointwise() const {
        return kh == 1 && kw == 1 && sh == 1 && sw == 1 && pt == 0 && pl == 0 && out_h == in_h && out_w == in_w &&
               (uint64_t)batch * plane() < ((uint64_t)1 << 31);
    }
    // and no y pattern: the images fold into the GEMM's columns (one slice of batch * plane lines)
    bool fold() const { return pointwise() && cn == 0 && cs == plane(); }
};

// The 1x1 convolutions whose waves take their operand straight from the pixels (conv_point*_kernel)
// instead of the fold split and the plane GEMM: up to 64 input channels at any output, as a wave keeps
// its pixels; otherwise, as every row tile splits the input again and each wave loads its own weights,
// up to 1280 output channels and 2^19 weights, or two tiles a compute unit.  Measured us (both launches
// of the other form): 24 -> 144 at 32 x 56 x 56 16.9 (46.8), 64 -> 256 at 16 x 56 x 56 17.1 (35.2), 960 -> 320 at
// 32 x 7 x 7 11.9 (17.9), 512 -> 512 at 32 x 28 x 28 59.2 (71.9), 320 -> 1280 at 32 x 7 x 7 13.6 (13.7), 2048 -> 1000
// at 1 x 7 x 7 9.7 (19.6); 512 -> 1024 at 32 x 7 x 7 16.1 (15.0), 2048 -> 512 at 32 x 7 x 7 28.8 (25.1).
bool point_path(const ConvGeom& g, const DeviceState* st) {
    if (!g.pointwise() || 2ull * g.in_ch * g.plane() > 0xFFFFFFFFull) return false;
    if (g.in_ch <= 64) return true;
    const uint64_t tiles = (uint64_t)ceil_div(g.out_ch, 32) * ceil_div((size_t)g.batch * g.plane(), 32);
    return (g.out_ch <= 1280 && (uint64_t)g.in_ch * g.out_ch < (1u << 19)) || tiles <= 2ull * st->cus;
}

int point_launch(const int16_t* x, const Planes& A, const int16_t* bptr, int16_t* y, const ConvGeom& g, uint32_t batch,
                  const DeviceState* st, hipStream_t s, int32_t lo, int32_t hi) {
    const uint32_t plane = g.plane(), k = g.in_ch, cols = batch * plane, tr = ceil_div(g.out_ch, 32), tc = ceil_div(cols, 32);
    const EpiConv epi{y, bptr, (uint64_t)g.out_ch * plane, g.out_ch, plane, g.cs, g.cn, g.gs, g.wrap, 0, 0, lo, hi};
    const uint32_t mode = g.wrap ? kWrap : (k <= 256 ? kSatTiny : (k <= 8192 ? kSatNarrow : kSatWide));
    const bool rag = k % 16 != 0;
    const uint64_t tiles = (uint64_t)tr * tc, cus = st->cus;
    if (k <= 64) {
        // up to 3 row tiles a wave while two waves a SIMD remain (24 -> 144 at 32 x 56 x 56: 1 / 2 / 3 / 4 tiles
        // 19.2 / 17.0 / 17.1 / 19.9 us; 64 -> 384 at 32 x 14 x 14, 2352 tiles: 6.3 / 7.1 / 7.4)
        const uint32_t gt = (uint32_t)std::min<uint64_t>({kPointTiles, tr, std::max<uint64_t>(1, tiles / (8 * cus))});
        const uint32_t br = ceil_div(tr, gt), bc = ceil_div(tc, 4);
#define CM_WIDE(NK_, RAG_)                                                                                               \
    CM_LAUNCH("conv_point_kernel", (conv_point_wide_kernel<NK_, RAG_>), dim3(br * bc), dim3(256), 0, s, A.hi, A.lo, \
              A.part, x, k, plane, cols, br, bc, tr, gt, A.kp, mode, epi)
        if (k <= 32) {
            if (rag) { CM_WIDE(1, true); } else { CM_WIDE(1, false); }
        } else {
            if (rag) { CM_WIDE(2, true); } else { CM_WIDE(2, false); }
        }
#undef CM_WIDE
        return CM_OK;
    }
    // two pixels a lane where that leaves three waves a compute unit (256 -> 256 at 8 x 28 x 28, 784 tiles of
    // 64 pixels: 8.5 us against 10.0), else one: alone from 4 waves a unit up (160 -> 960 at 32 x 7 x 7, 1470
    // tiles: 8.2 / 8.2 / 9.5 with 1 / 2 / 4 waves), two of them sharing the channels from 2.5 up (512 -> 512 at
    // 8 x 14 x 14, 784 tiles: 10.6 / 10.1 / 10.9), four below (576 -> 160 at 32 x 7 x 7, 245 tiles: 8.4 / 6.7 / 6.3)
#define CM_POINT1(PX_, KW_, RAG_)                                                                                        \
    CM_LAUNCH("conv_point_kernel", (conv_point_kernel<PX_, KW_, RAG_>), dim3(tr * ceil_div(cols, 32 * PX_)), dim3(64 * KW_), \
              0, s, A.hi, A.lo, A.part, A.lines_p, A.nsum(), x, k, plane, cols, tr, ceil_div(cols, 32 * PX_), A.kp, mode, epi)
#define CM_POINT(PX_, KW_) \
    if (rag) { CM_POINT1(PX_, KW_, true); } else { CM_POINT1(PX_, KW_, false); }
    if (plane % 2 == 0 && (uint64_t)tr * ceil_div(cols, 64) >= 3 * cus) { CM_POINT(2, 1) }
    else if (tiles >= 4 * cus) { CM_POINT(1, 1) }
    else if (2 * tiles >= 5 * cus) { CM_POINT(1, 2) }
    else { CM_POINT(1, 4) }
#undef CM_POINT
#undef CM_POINT1
    return CM_OK;
}

// k of the GEMM: 16-channel tiles x kernel positions (the packed weight order), in BK steps.
uint32_t conv_kp(uint32_t in_ch, uint32_t kh, uint32_t kw) {
    return (uint32_t)round_up((uint64_t)((in_ch + 15) / 16) * kh * kw * 16, BK);
}

Planes conv_b_planes(const ConvGeom& g, uint32_t kp) {
    return g.fold() ? make_planes(g.batch * g.plane(), kp, 1) : make_planes(g.plane(), kp, g.batch);
}

GemmPlan conv_plan(const ConvGeom& g, const Planes& B, const DeviceState* st) {
    return gemm_plan(g.out_ch, B.rows, B.slices, B.kp / BK, false, st->cus);
}

// The weights' planes: rows = output channels in the packed tile-major order (ConvKernel.h:136-159).
int conv_split_w(const int16_t* w, Planes& A, uint32_t out_ch, uint32_t in_ch, uint32_t kh, uint32_t kw,
                 hipStream_t s) {
    const uint32_t tiles = (in_ch + 15) / 16;
    const uint32_t rem = in_ch - (tiles - 1) * 16, last = rem <= 8 ? 8 : 16;
    const uint32_t per_m = kh * kw * ((tiles - 1) * 16 + last);
    return run_split<SrcConvW, true>(SrcConvW{w, out_ch, in_ch, kh, kw, tiles, per_m, last}, 0, A, s);
}

// A 1x1 convolution from its pixels with the weights' planes A (point_path): no planes of the input.
int conv_point(const int16_t* x, const Planes& A, const int16_t* bptr, int16_t* y, const ConvGeom& g,
               const DeviceState* st, hipStream_t s, int32_t lo, int32_t hi) {
    const uint32_t plane = g.plane();
    // images whose input stays below the kernels' 32-bit byte offsets, one launch each
    const uint32_t per = (uint32_t)std::min<uint64_t>(g.batch, 0xFFFFFFFFull / (2ull * g.in_ch * plane));
    for (uint32_t i = 0; i < g.batch; i += per) {
        const int rc = point_launch(x + (uint64_t)i * g.in_ch * plane, A, bptr, y + (uint64_t)i * g.out_ch * plane, g,
                                    std::min(per, g.batch - i), st, s, lo, hi);
        if (rc) return rc;
    }
    return CM_OK;
}

// The input's planes (im2col, or the folded 1x1 form) and the GEMM with the weights' planes A.
int conv_gemm(const int16_t* x, const Planes& A, Planes& B, const int16_t* bptr, int16_t* y, const ConvGeom& g,
              const DeviceState* st, hipStream_t s, int32_t lo, int32_t hi) {
    const uint32_t plane = g.plane();
    const uint64_t img = (uint64_t)g.out_ch * plane;
    if (g.fold()) {
        const uint32_t cols = g.batch * plane;
        if (B.lines_p / 64 >= 4 * st->cus) {
            // lines enough for the workgroups of whole slabs to fill the chip
            CM_LAUNCH("split_fold_kernel", split_fold_lds_kernel, dim3(B.lines_p / 64, B.nslab), dim3(256), 0, s, x,
                      g.in_ch, plane, (uint64_t)g.in_ch * plane, cols, B.hi, B.lo, B.part, B.lines_p, B.kp);
        } else if (B.lines_p / 64 >= (uint32_t)st->cus) {
            // one wave per 64 k of the slab
            const uint32_t waves = std::min<uint32_t>(16, ceil_div(std::min<uint32_t>(B.kp, SLAB), 64));
            CM_LAUNCH("split_fold_kernel", split_fold_kernel, dim3(B.lines_p / 64, B.nslab), dim3(64 * waves), 0, s,
                      x, g.in_ch, plane, (uint64_t)g.in_ch * plane, cols, B.hi, B.lo, B.part, B.lines_p, B.kp);
        } else {
            // few lines: 16 a workgroup
            const uint32_t waves = std::min<uint32_t>(16, ceil_div(std::min<uint32_t>(B.kp, SLAB), 64));
            CM_LAUNCH("split_fold_kernel", split_fold16_kernel, dim3(B.lines_p / 16, B.nslab), dim3(64 * waves), 0,
                      s, x, g.in_ch, plane, (uint64_t)g.in_ch * plane, cols, B.hi, B.lo, B.part, B.lines_p, B.kp);
        }
        const bool pairs = (reinterpret_cast<uintptr_t>(y) & 3) == 0 && (plane & 1) == 0;
        EpiConv epi{y, bptr, img, g.out_ch, cols, plane, 0, 0, g.wrap, pairs ? 1u : 0u, plane, lo, hi};
        return run_gemm(A, B, 1, g.in_ch * g.kh * g.kw, epi, s);
    }
    const Im2col im{x, (uint64_t)g.in_ch * g.in_h * g.in_w, g.in_ch, g.in_h, g.in_w, g.out_w, g.kh, g.kw, g.sh, g.sw,
                    g.dh, g.dw, g.pt, g.pl, plane};
    const uint32_t waves = std::min<uint32_t>(16, ceil_div(std::min<uint32_t>(B.kp, SLAB), 64));
    CM_LAUNCH("split_kernel", split_im2col_kernel, dim3(B.lines_p / 16, B.nslab, B.slices), dim3(64 * waves), 0, s, im,
              B.hi, B.lo, B.part, B.lines_p, B.kp, B.nslab);
    const bool pairs = (reinterpret_cast<uintptr_t>(y) & 3) == 0 && (plane & 1) == 0 && (g.cs & 1) == 0 &&
                       (g.gs & 1) == 0 && (img & 1) == 0;
    EpiConv epi{y, bptr, img, g.out_ch, plane, g.cs, g.cn, g.gs, g.wrap, pairs ? 1u : 0u, 0, lo, hi};
    return run_gemm(A, B, g.batch, g.in_ch * g.kh * g.kw, epi, s);
}

// The output bounds of a fused activation (the VectorOP act codes RELU = 1, RELU6 = 2, applied
// to the raw int16 result: VectorOP ops 4 and 5 on the conv's output); CM_EINVAL otherwise.
int act_bounds(uint32_t act, int32_t& lo, int32_t& hi) {
    lo = -32768;
    hi = 32767;
    if (act == 0) return CM_OK;
    if (act == 1 || act == 2) {
        lo = 0;
        if (act == 2) hi = 6 << 8;
        return CM_OK;
    }
    return fail(CM_EINVAL, "conv: act %u (0 none, 1 RELU, 2 RELU6)", act);
}

}  // namespace
}  // namespace cm

namespace cm {
namespace {

int conv_run(const int16_t* x, const int16_t* w, const int16_t* bias, int16_t* y, uint32_t batch, uint32_t in_ch,
             uint32_t in_h, uint32_t in_w, uint32_t out_ch, uint32_t out_h, uint32_t out_w, uint32_t kh, uint32_t kw,
             uint32_t stride_h, uint32_t stride_w, uint32_t dilation_h, uint32_t dilation_w, uint32_t pad_top,
             uint32_t pad_left, uint32_t has_bias, uint32_t is_depthwise, uint32_t y_cs, uint32_t y_cn,
             uint32_t y_gs, uint32_t wrap32, uint32_t act, void* stream) {
    DeviceState* st;
    int rc = state(&st);
    if (rc) return rc;
    int32_t lo, hi;
    rc = act_bounds(act, lo, hi);
    if (rc) return rc;
    if (batch == 0 || out_ch == 0 || out_h == 0 || out_w == 0) return CM_OK;
    if (kh == 0 || kw == 0 || kh > 7 || kw > 7) return fail(CM_EINVAL, "conv: kernel %ux%u outside 1..7", kh, kw);
    if (stride_h == 0 || stride_w == 0 || dilation_h == 0 || dilation_w == 0)
        return fail(CM_EINVAL, "conv: zero stride or dilation");
    if ((y_cs || y_cn) && batch != 1) return fail(CM_EINVAL, "conv: y pattern needs batch 1");
    if (is_depthwise && in_ch != out_ch) return fail(CM_EINVAL, "conv: depthwise in_ch %u != out_ch %u", in_ch, out_ch);
    if (in_ch == 0) return fail(CM_EINVAL, "conv: in_ch 0");
    hipStream_t s = as_stream(stream);
    const uint32_t plane = out_h * out_w;
    const uint32_t cs = y_cs ? y_cs : plane;
    const int16_t* bptr = has_bias ? bias : nullptr;
    const bool dw3 = is_depthwise && kh == 3 && kw == 3 && dilation_h == 1 && dilation_w == 1;
    if (dw3 && stride_h == 1 && stride_w == 1 && pad_left <= 2 && (in_w & 7) == 0 && (out_w & 7) == 0 &&
        aligned16(x) && aligned16(y) && (cs & 7) == 0 && (!y_cn || (y_gs & 7) == 0)) {
        constexpr uint32_t R = 4;
        const uint32_t strips = (out_h + R - 1) / R, groups = out_w / 8;
        const uint64_t items = (uint64_t)batch * out_ch * strips * groups;
        if (items < ((uint64_t)1 << 31)) {
            const unsigned blocks = (unsigned)std::min<uint64_t>((items + 255) / 256, 65536ull * 8);
#define CM_DW3V(PL)                                                                                              \
    CM_LAUNCH("conv_dw3v_kernel", (conv_dw3v_kernel<PL, R>), dim3(blocks), dim3(256), 0, s, x, w, bptr, y,       \
              (uint32_t)items, strips, groups, out_ch, in_h, in_w, out_h, out_w, pad_top, 16u, cs, y_cn, y_gs, \
              wrap32 ? 1u : 0u, lo, hi)
            if (pad_left == 0) { CM_DW3V(0); }
            else if (pad_left == 1) { CM_DW3V(1); }
            else { CM_DW3V(2); }
#undef CM_DW3V
            return CM_OK;
        }
    }
    if (dw3 && stride_h == stride_w && stride_h <= 2) {
        // Lanes a unit up to which the strips win, from both kernels over 9 plane counts of 45 shapes (us, and
        // conv_dw3_kernel's): one workgroup, 2048 planes of 7 x 7 4.0 (4.2), 12288 at 1.3 4.65 (4.49); more over
        // rows that fill less than half of a lane's 10 columns (12288 of 12 x 3 3.9 and 5.2, 61440 of 40 x 3 12
        // % behind), any over rows of 4 at stride 1 (131072 of 20 x 4 20.9 and 24.4) and over planes of at most
        // 5 x 5 (30720 of 3 x 3 4.2 and 5.4; 131072 of 5 x 5 4 % behind); none at stride 2 over rows of 4 or 8
        // columns in whole strips (2048 of 8 x 8 5.4 and 4.6)
        uint64_t most = 256;
        if ((in_w <= 5 && in_h <= 5) || (in_w == 4 && stride_h == 1)) most = (1ull << 31) / st->cus;
        else if (stride_h == 2 && (in_w == 4 || in_w == 8) && out_h % 4 == 0) most = 0;
        else if (in_w <= 3) most = stride_h == 1 ? 1200 : 512;
        const uint32_t R = stride_h == 1 ? 8 : 4, strips = ceil_div(out_h, R);
        const uint64_t items = (uint64_t)batch * out_ch * strips * out_w;
        if (items < (1ull << 31) && items <= most * st->cus) {
#define CM_DW3S(S_, R_)                                                                                         \
    CM_LAUNCH("conv_dw3_kernel", (conv_dw3_strip_kernel<S_, R_>), dim3(std::min(ceil_div(items, 256), 65536u * 8)), dim3(256), 0, s, x, w, \
              bptr, y, (uint32_t)items, strips, out_ch, in_h, in_w, out_h, out_w, pad_top, pad_left, 16u, cs, y_cn, y_gs, \
              wrap32 ? 1u : 0u, lo, hi)
            if (stride_h == 1) { CM_DW3S(1, 8); } else { CM_DW3S(2, 4); }
#undef CM_DW3S
            return CM_OK;
        }
    }
    if (dw3 && stride_h == stride_w && stride_h <= 2 && (uint64_t)in_h * in_w < (1u << 29) &&
        (uint64_t)batch * out_ch * in_h * in_w >= 10 && out_h < (1u << 27) && out_w < (1u << 27) &&
        pad_top < (1u << 28) && pad_left < (1u << 28) && (uint64_t)batch * out_ch < (1u << 31)) {
        constexpr uint32_t R = 2;
        const uint32_t strips = ceil_div(out_h, R), groups = ceil_div((size_t)out_w * stride_w, 8);
        const uint64_t items = (uint64_t)batch * out_ch * strips * groups;
        if (items < ((uint64_t)1 << 31)) {
            const unsigned blocks = (unsigned)std::min<uint64_t>((items + 255) / 256, 65536ull * 8);
#define CM_DW3(S_)                                                                                              \
    CM_LAUNCH("conv_dw3_kernel", (conv_dw3_kernel<S_, R>), dim3(blocks), dim3(256), 0, s, x, w, bptr, y, (uint32_t)items, \
              batch * out_ch, strips, groups, out_ch, in_h, in_w, out_h, out_w, pad_top, pad_left, 16u, cs, y_cn, y_gs, \
              wrap32 ? 1u : 0u, lo, hi)
            if (stride_h == 1) { CM_DW3(1); } else { CM_DW3(2); }
#undef CM_DW3
            return CM_OK;
        }
    }
    if (is_depthwise) {
        const uint64_t total = (uint64_t)batch * out_ch * plane;
        uint64_t blocks = (total + 255) / 256;
        if (blocks > 65536ull * 8) blocks = 65536ull * 8;
        CM_LAUNCH("conv_dw_kernel", conv_dw_kernel, dim3((unsigned)blocks), dim3(256), 0, s, x, w, bptr, y, total,
                           out_ch, in_h, in_w, out_h, out_w, kh, kw, stride_h, stride_w, dilation_h,
                           dilation_w, pad_top, pad_left, (kh * kw + 7) & ~7u, cs, y_cn, y_gs,
                           wrap32 ? 1u : 0u, lo, hi);
        return CM_OK;
    }
    if (in_ch * kh * kw <= kCsMaxTaps && (uint64_t)in_ch * kh * kw * out_ch <= kCsMaxWork && batch <= 65535 &&
        (uint64_t)in_ch * in_h * in_w < (1ull << 31) && kh <= 32 && kw <= 32 &&
        (uint64_t)out_h * stride_h * in_w + (uint64_t)out_w * stride_w < (1ull << 31)) {
        // few taps: straight on the VALU
        const uint32_t taps = in_ch * kh * kw, tiles = (in_ch + 15) / 16;
        const uint32_t rem = in_ch - (tiles - 1) * 16, last = rem <= 8 ? 8u : 16u;
        const uint32_t np = (uint32_t)round_up(ceil_div(taps, 2), 4);
        // output channels a workgroup: 32 over planes of at least 56 x 56 (the pixels' taps
        // loaded once for more channels), 16 below, 4 where 16 would leave most compute units
        // idle (a small CNN's 14 x 14 planes at batch 1)
        const uint64_t pblocks = (uint64_t)ceil_div(plane, 256) * batch;
        const uint32_t og = pblocks * ceil_div(out_ch, 16) < (uint64_t)st->cus ? 4u : (plane >= 3136 ? 32u : 16u);
        const ConvSmall cv{x, w, bptr, y, in_ch, in_h, in_w, out_ch, out_h, out_w, kh, kw, stride_h, stride_w,
                           dilation_h, dilation_w, pad_top, pad_left, kh * kw * ((tiles - 1) * 16 + last), tiles, last,
                           cs, y_cn, y_gs, wrap32 ? 1u : 0u, lo, hi, og};
        const dim3 grid(ceil_div(plane, 256), ceil_div(out_ch, og), batch);
        const bool pw = kh == 1 && kw == 1 && stride_h == 1 && stride_w == 1 && pad_top == 0 && pad_left == 0 &&
                        in_h == out_h && in_w == out_w;
#define CM_CS(NP_)                                                                                              \
    case NP_:                                                                                                   \
        if (pw) { CM_LAUNCH("conv_small_kernel", (conv_small_kernel<NP_, true>), grid, dim3(256), 0, s, cv); }   \
        else { CM_LAUNCH("conv_small_kernel", (conv_small_kernel<NP_, false>), grid, dim3(256), 0, s, cv); }     \
        return CM_OK;
        switch (np) {
            CM_CS(4) CM_CS(8) CM_CS(12) CM_CS(16) CM_CS(20) CM_CS(24) CM_CS(28) CM_CS(32) CM_CS(36) CM_CS(40)
        default: break;
        }
#undef CM_CS
    }
    if ((uint64_t)in_ch * kh * kw > 32768)
        return fail(CM_EINVAL, "conv: in_ch * kh * kw = %u above 32768", in_ch * kh * kw);
    const ConvGeom g{batch, in_ch, in_h, in_w, out_ch, out_h, out_w, kh, kw, stride_h, stride_w, dilation_h,
                     dilation_w, pad_top, pad_left, cs, y_cn, y_gs, wrap32 ? 1u : 0u};
    const uint32_t kp = conv_kp(in_ch, kh, kw);
    const bool point = point_path(g, st);
    Planes B = point ? Planes{} : conv_b_planes(g, kp);
    Planes A = point ? make_planes(out_ch, kp, 1) : make_a_planes(out_ch, kp, 1, conv_plan(g, B, st));
    void* ws;
    rc = workspace(st, A.bytes() + (point ? 0 : B.bytes()), &ws, s);
    if (rc) return rc;
    char* p = static_cast<char*>(ws);
    A.carve(p);
    rc = conv_split_w(w, A, out_ch, in_ch, kh, kw, s);
    if (rc) return rc;
    if (point) return conv_point(x, A, bptr, y, g, st, s, lo, hi);
    B.carve(p);
    return conv_gemm(x, A, B, bptr, y, g, st, s, lo, hi);
}

}  // namespace
}  // namespace cm

extern "C" int cm_conv(const int16_t* x, const int16_t* w, const int16_t* bias, int16_t* y,
                       uint32_t batch, uint32_t in_ch, uint32_t in_h, uint32_t in_w, uint32_t out_ch,
                       uint32_t out_h, uint32_t out_w, uint32_t kh, uint32_t kw, uint32_t stride_h,
                       uint32_t stride_w, uint32_t dilation_h, uint32_t dilation_w, uint32_t pad_top,
                       uint32_t pad_left, uint32_t has_bias, uint32_t is_depthwise, uint32_t y_cs,
                       uint32_t y_cn, uint32_t y_gs, uint32_t wrap32, void* stream) {
    return cm::conv_run(x, w, bias, y, batch, in_ch, in_h, in_w, out_ch, out_h, out_w, kh, kw, stride_h, stride_w,
                        dilation_h, dilation_w, pad_top, pad_left, has_bias, is_depthwise, y_cs, y_cn, y_gs, wrap32,
                        0, stream);
}

extern "C" int cm_conv_act(const int16_t* x, const int16_t* w, const int16_t* bias, int16_t* y, uint32_t batch,
                           uint32_t in_ch, uint32_t in_h, uint32_t in_w, uint32_t out_ch, uint32_t out_h,
                           uint32_t out_w, uint32_t kh, uint32_t kw, uint32_t stride_h, uint32_t stride_w,
                           uint32_t dilation_h, uint32_t dilation_w, uint32_t pad_top, uint32_t pad_left,
                           uint32_t has_bias, uint32_t is_depthwise, uint32_t y_cs, uint32_t y_cn, uint32_t y_gs,
                           uint32_t wrap32, uint32_t act, void* stream) {
    return cm::conv_run(x, w, bias, y, batch, in_ch, in_h, in_w, out_ch, out_h, out_w, kh, kw, stride_h, stride_w,
                        dilation_h, dilation_w, pad_top, pad_left, has_bias, is_depthwise, y_cs, y_cn, y_gs, wrap32,
                        act, stream);
}

extern "C" size_t cm_conv_w_planes_bytes(uint32_t out_ch, uint32_t in_ch, uint32_t kh, uint32_t kw) {
    using namespace cm;
    if (out_ch == 0 || in_ch == 0 || kh == 0 || kw == 0) return 0;
    return make_planes(out_ch, conv_kp(in_ch, kh, kw), 1, 256).bytes();
}

extern "C" int cm_conv_split_w(const int16_t* w, void* planes, uint32_t out_ch, uint32_t in_ch, uint32_t kh,
                               uint32_t kw, void* stream) {
    using namespace cm;
    DeviceState* st;
    int rc = state(&st);
    if (rc) return rc;
    if (out_ch == 0) return CM_OK;
    if (in_ch == 0 || kh == 0 || kw == 0 || kh > 7 || kw > 7) return fail(CM_EINVAL, "conv: weights %ux%ux%u", in_ch, kh, kw);
    if ((uint64_t)in_ch * kh * kw > 32768)
        return fail(CM_EINVAL, "conv: in_ch * kh * kw = %u above 32768", in_ch * kh * kw);
    if (reinterpret_cast<uintptr_t>(planes) & 255) return fail(CM_EALIGN, "conv: weight planes not 256-byte aligned");
    Planes A = make_planes(out_ch, conv_kp(in_ch, kh, kw), 1, 256);
    char* p = static_cast<char*>(planes);
    A.carve(p);
    return conv_split_w(w, A, out_ch, in_ch, kh, kw, as_stream(stream));
}

namespace cm {
namespace {

int conv_planes_run(const int16_t* x, const void* w_planes, const int16_t* bias, int16_t* y, uint32_t batch,
                    uint32_t in_ch, uint32_t in_h, uint32_t in_w, uint32_t out_ch, uint32_t out_h, uint32_t out_w,
                    uint32_t kh, uint32_t kw, uint32_t stride_h, uint32_t stride_w, uint32_t dilation_h,
                    uint32_t dilation_w, uint32_t pad_top, uint32_t pad_left, uint32_t has_bias,
                    uint32_t is_depthwise, uint32_t y_cs, uint32_t y_cn, uint32_t y_gs, uint32_t wrap32,
                    uint32_t act, void* stream) {
    DeviceState* st;
    int rc = state(&st);
    if (rc) return rc;
    int32_t lo, hi;
    rc = act_bounds(act, lo, hi);
    if (rc) return rc;
    if (batch == 0 || out_ch == 0 || out_h == 0 || out_w == 0) return CM_OK;
    if (is_depthwise) return fail(CM_EINVAL, "conv: weight planes are for standard convolutions");
    if (kh == 0 || kw == 0 || kh > 7 || kw > 7) return fail(CM_EINVAL, "conv: kernel %ux%u outside 1..7", kh, kw);
    if (stride_h == 0 || stride_w == 0 || dilation_h == 0 || dilation_w == 0)
        return fail(CM_EINVAL, "conv: zero stride or dilation");
    if ((y_cs || y_cn) && batch != 1) return fail(CM_EINVAL, "conv: y pattern needs batch 1");
    if (in_ch == 0) return fail(CM_EINVAL, "conv: in_ch 0");
    if ((uint64_t)in_ch * kh * kw > 32768)
        return fail(CM_EINVAL, "conv: in_ch * kh * kw = %u above 32768", in_ch * kh * kw);
    if (reinterpret_cast<uintptr_t>(w_planes) & 255) return fail(CM_EALIGN, "conv: weight planes not 256-byte aligned");
    hipStream_t s = as_stream(stream);
    const uint32_t plane = out_h * out_w;
    const ConvGeom g{batch, in_ch, in_h, in_w, out_ch, out_h, out_w, kh, kw, stride_h, stride_w, dilation_h,
                     dilation_w, pad_top, pad_left, y_cs ? y_cs : plane, y_cn, y_gs, wrap32 ? 1u : 0u};
    const uint32_t kp = conv_kp(in_ch, kh, kw);
    const int16_t* bptr = has_bias ? bias : nullptr;
    Planes A = make_planes(out_ch, kp, 1, 256);
    char* q = static_cast<char*>(const_cast<void*>(w_planes));
    A.carve(q);
    if (point_path(g, st)) return conv_point(x, A, bptr, y, g, st, s, lo, hi);
    Planes B = conv_b_planes(g, kp);
    A.plan = conv_plan(g, B, st);
    void* ws;
    rc = workspace(st, B.bytes(), &ws, s);
    if (rc) return rc;
    char* p = static_cast<char*>(ws);
    B.carve(p);
    return conv_gemm(x, A, B, bptr, y, g, st, s, lo, hi);
}

}  // namespace
}  // namespace cm

extern "C" int cm_conv_planes(const int16_t* x, const void* w_planes, const int16_t* bias, int16_t* y,
                              uint32_t batch, uint32_t in_ch, uint32_t in_h, uint32_t in_w, uint32_t out_ch,
                              uint32_t out_h, uint32_t out_w, uint32_t kh, uint32_t kw, uint32_t stride_h,
                              uint32_t stride_w, uint32_t dilation_h, uint32_t dilation_w, uint32_t pad_top,
                              uint32_t pad_left, uint32_t has_bias, uint32_t is_depthwise, uint32_t y_cs,
                              uint32_t y_cn, uint32_t y_gs, uint32_t wrap32, void* stream) {
    return cm::conv_planes_run(x, w_planes, bias, y, batch, in_ch, in_h, in_w, out_ch, out_h, out_w, kh, kw, stride_h,
                               stride_w, dilation_h, dilation_w, pad_top, pad_left, has_bias, is_depthwise, y_cs,
                               y_cn, y_gs, wrap32, 0, stream);
}

extern "C" int cm_conv_planes_act(const int16_t* x, const void* w_planes, const int16_t* bias, int16_t* y,
                                  uint32_t batch, uint32_t in_ch, uint32_t in_h, uint32_t in_w, uint32_t out_ch,
                                  uint32_t out_h, uint32_t out_w, uint32_t kh, uint32_t kw, uint32_t stride_h,
                                  uint32_t stride_w, uint32_t dilation_h, uint32_t dilation_w, uint32_t pad_top,
                                  uint32_t pad_left, uint32_t has_bias, uint32_t is_depthwise, uint32_t y_cs,
                                  uint32_t y_cn, uint32_t y_gs, uint32_t wrap32, uint32_t act, void* stream) {
    return cm::conv_planes_run(x, w_planes, bias, y, batch, in_ch, in_h, in_w, out_ch, out_h, out_w, kh, kw, stride_h,
                               stride_w, dilation_h, dilation_w, pad_top, pad_left, has_bias, is_depthwise, y_cs,
                               y_cn, y_gs, wrap32, act, stream);
}

extern "C" int cm_matmul_strided(const int16_t* a, const int16_t* b, int16_t* c, uint32_t n, uint32_t k, uint32_t m,
                                 uint32_t batch, uint32_t inner, uint64_t lda, uint64_t a_bs, uint64_t a_bs2,
                                 uint64_t ldb, uint64_t b_bs, uint64_t b_bs2, uint32_t b_trans, uint64_t ldc,
                                 uint64_t c_bs, uint64_t c_bs2, uint32_t wrap32, void* stream) {
    using namespace cm;
    DeviceState* st;
    int rc = state(&st);
    if (rc) return rc;
    if (n == 0 || m == 0 || batch == 0) return CM_OK;
    if (k == 0 || k > 32768) return fail(CM_EINVAL, "matmul: k = %u outside 1 .. 32768", k);
    if (inner == 0) return fail(CM_EINVAL, "matmul: inner 0");
    const bool a_ok = aligned16(a) && (lda & 7) == 0 && (a_bs & 7) == 0 && (a_bs2 & 7) == 0 && (k & 7) == 0;
    const bool b_ok = aligned16(b) && (ldb & 7) == 0 && (b_bs & 7) == 0 && (b_bs2 & 7) == 0 &&
                      (b_trans ? (k & 7) == 0 : (m & 7) == 0);
    if (!a_ok || !b_ok) return fail(CM_EALIGN, "matmul: strided operands need 16-byte rows and slices");
    if (lda < k || ldb < (b_trans ? k : m) || ldc < m) return fail(CM_EINVAL, "matmul: row strides below the rows");
    hipStream_t s = as_stream(stream);
    const uint32_t kp = (uint32_t)round_up(k, BK);
    Planes A = make_a_planes(n, kp, batch, gemm_plan(n, m, batch, kp / BK, false, st->cus)), B = make_planes(m, kp, batch);
    void* ws;
    rc = workspace(st, A.bytes() + B.bytes(), &ws, s);
    if (rc) return rc;
    char* p = static_cast<char*>(ws);
    A.carve(p);
    B.carve(p);
    rc = split_row_lines(a, Slices{a_bs, a_bs2, inner}, lda, n, k, A, s);
    if (rc) return rc;
    if (b_trans) {
        rc = split_row_lines(b, Slices{b_bs, b_bs2, inner}, ldb, m, k, B, s);
        if (rc) return rc;
    } else {
        CM_LAUNCH("split_cols_kernel", split_cols_kernel, dim3(B.lines_p / 32, B.nslab, B.slices), dim3(256), 0, s,
                  b, (Slices{b_bs, b_bs2, inner}), ldb, 0u, m, k, B.hi, B.lo, B.part, B.lines_p, B.kp, B.nslab);
    }
    const bool pairs = (reinterpret_cast<uintptr_t>(c) & 3) == 0 && (m & 1) == 0 && (ldc & 1) == 0 &&
                       (c_bs & 1) == 0 && (c_bs2 & 1) == 0;
    EpiMatmul epi{c, c_bs, n, m, wrap32 ? 1u : 0u, pairs ? 1u : 0u, ldc, c_bs2, inner};
    return run_gemm(A, B, batch, k, epi, s);
}

extern "C" int cm_matmul_skinny_multi(const int16_t* a, uint32_t n, uint32_t k, uint32_t count,
                                      const int16_t* const* b, int16_t* const* c, const uint32_t* m,
                                      uint32_t b_packed, void* stream) {
    using namespace cm;
    DeviceState* st;
    int rc = state(&st);
    if (rc) return rc;
    if (count == 0 || count > kSkinnySegs) return fail(CM_EINVAL, "matmul: %u products (1 .. %u)", count, kSkinnySegs);
    if (n == 0) return CM_OK;
    if (n > 32 || k == 0 || k > 32768 || (k & 1) || b_packed > 2 || (b_packed == 2 && (k & 7)))
        return fail(CM_EINVAL, "matmul: skinny products take n <= 32, even k <= 32768 (k %% 8 == 0 transposed)");
    if (reinterpret_cast<uintptr_t>(a) & 3) return fail(CM_EALIGN, "matmul: a not 4-byte aligned");
    for (uint32_t i = 0; i < count; i++) {
        if (m[i] == 0 || (m[i] & 1) || (b_packed == 1 && (m[i] & 31)))
            return fail(CM_EINVAL, "matmul: product %u: m = %u", i, m[i]);
        if ((reinterpret_cast<uintptr_t>(b[i]) & (b_packed == 2 ? 15 : 3)) || (reinterpret_cast<uintptr_t>(c[i]) & 3))
            return fail(CM_EALIGN, "matmul: product %u: b / c not aligned", i);
    }
    return skinny_run(a, n, k, 1, 0, 0, 0, count, b, c, m, b_packed, st, as_stream(stream));
}

namespace cm {
namespace {

// 16-column blocks a skinny workgroup owns, for a launch of blocks16 blocks over k.
uint32_t skinny_blocks(uint64_t blocks16, uint32_t k) {
    (void)k;
    return blocks16 >= 2048 ? 4u : (blocks16 >= 256 ? 2u : 1u);
}

// The segments of a skinny launch (checked, the planes carved), the slabs of their column sums
// and the 16-column blocks they hold.
int skinny_segs(uint32_t n, uint32_t k, uint32_t count, const int16_t* a, const void* const* b_planes,
                int16_t* const* c, const uint32_t* m, SkinnyPlaneSegs& segs, uint32_t& nslab, uint64_t& blocks16) {
    if (count == 0 || count > kSkinnySegs) return fail(CM_EINVAL, "matmul: %u products (1 .. %u)", count, kSkinnySegs);
    if (n > 16 || k == 0 || k > 32768 || (k & 7))
        return fail(CM_EINVAL, "matmul: skinny plane products take n <= 16 and k a multiple of 8 up to 32768");
    if (!aligned16(a)) return fail(CM_EALIGN, "matmul: a not 16-byte aligned");
    const uint32_t kp = (uint32_t)round_up(k, BK);
    segs = SkinnyPlaneSegs{};
    segs.count = count;
    blocks16 = 0;
    nslab = 0;
    for (uint32_t i = 0; i < count; i++) {
        if (m[i] == 0) return fail(CM_EINVAL, "matmul: product %u: m = 0", i);
        if (reinterpret_cast<uintptr_t>(b_planes[i]) & 255)
            return fail(CM_EALIGN, "matmul: product %u: b planes not 256-byte aligned", i);
        Planes B = make_planes(m[i], kp, 1);
        char* q = static_cast<char*>(const_cast<void*>(b_planes[i]));
        B.carve(q);
        segs.hi[i] = B.hi;
        segs.lo[i] = B.lo;
        segs.part[i] = B.part;
        segs.c[i] = c[i];
        segs.m[i] = m[i];
        segs.lines_p[i] = B.lines_p;
        nslab = B.nslab;
        blocks16 += ceil_div(m[i], 16);
    }
    return CM_OK;
}

// Wavefronts of an nb-block skinny workgroup over k (one round of loads where they allow) and
// the LDS of their partials.
uint32_t skinny_waves(uint32_t k, uint32_t nb) {
    const uint32_t kp = (uint32_t)round_up(k, BK);
    return std::min<uint32_t>(sp_max_waves(nb), std::max<uint32_t>(1, ceil_div(kp / 64, sp_chunk(nb))));
}
size_t skinny_lds(uint32_t waves, uint32_t nb, bool sat = false) {
    return (size_t)waves * 16 * (16 * nb * (sat ? 3 : 1) + 1) * 4;
}

int skinny_planes(const int16_t* a, uint32_t n, uint32_t k, uint32_t count, const void* const* b_planes,
                  int16_t* const* c, const uint32_t* m, const SkinnyAddx& ax, hipStream_t s, bool sat = false) {
    if (n == 0) return CM_OK;
    SkinnyPlaneSegs segs;
    uint32_t nslab;
    uint64_t blocks16;
    int rc = skinny_segs(n, k, count, a, b_planes, c, m, segs, nslab, blocks16);
    if (rc) return rc;
    const uint32_t kp = (uint32_t)round_up(k, BK);
    // the saturating partials take three times the LDS: at most two blocks a workgroup (50 KiB)
    const uint32_t nb = sat ? std::min<uint32_t>(2, skinny_blocks(blocks16, k)) : skinny_blocks(blocks16, k);
    uint64_t cbs = 0;
    for (uint32_t i = 0; i < count; i++) {
        segs.cb0[i] = (uint32_t)cbs;
        cbs += ceil_div(m[i], 16 * nb);
    }
    if (cbs > 0x7FFFFFFFull) return fail(CM_EINVAL, "matmul: %llu column blocks", (unsigned long long)cbs);
    const uint32_t waves = skinny_waves(k, nb);
    const size_t lds = skinny_lds(waves, nb, sat);
    const dim3 grid((uint32_t)cbs), block(64 * waves);
    const uint32_t xk = ax.out == nullptr ? 0u : (((ax.op >> 4) & 3) == 0 ? 1u : 2u);
    if (sat && xk) return fail(CM_EINVAL, "matmul: no output job on saturating skinny products");
#define CM_SP_LAUNCH(NB_, XK_)                                                                                  \
    CM_LAUNCH("skinny_planes_kernel", (skinny_planes_kernel<NB_, XK_>), grid, block, lds, s, a, n, k, kp, nslab, \
              segs, ax)
#define CM_SP_LAUNCH_SAT(NB_)                                                                                   \
    CM_LAUNCH("skinny_planes_kernel", (skinny_planes_kernel<NB_, 0, true>), grid, block, lds, s, a, n, k, kp,    \
              nslab, segs, ax)
    if (sat) {
        if (nb == 1) { CM_SP_LAUNCH_SAT(1); }
        else { CM_SP_LAUNCH_SAT(2); }
    } else if (xk == 0) {
        if (nb == 1) { CM_SP_LAUNCH(1, 0); }
        else if (nb == 2) { CM_SP_LAUNCH(2, 0); }
        else { CM_SP_LAUNCH(4, 0); }
    } else if (xk == 1) {
        if (nb == 1) { CM_SP_LAUNCH(1, 1); }
        else if (nb == 2) { CM_SP_LAUNCH(2, 1); }
        else { CM_SP_LAUNCH(4, 1); }
    } else {
        if (nb == 1) { CM_SP_LAUNCH(1, 2); }
        else if (nb == 2) { CM_SP_LAUNCH(2, 2); }
        else { CM_SP_LAUNCH(4, 2); }
    }
#undef CM_SP_LAUNCH
#undef CM_SP_LAUNCH_SAT
    return CM_OK;
}

int skinny_mulact(const int16_t* a, uint32_t n, uint32_t k, const void* b_gate, const void* b_up, int16_t* c_gate,
                  int16_t* c_up, uint32_t m, const SkinnyMulact& mj, hipStream_t s) {
    if (n == 0) return CM_OK;
    SkinnyPlaneSegs segs;
    uint32_t nslab;
    uint64_t blocks16;
    const void* bp[2] = {b_gate, b_up};
    int16_t* cp[2] = {c_gate, c_up};
    const uint32_t ms[2] = {m, m};
    int rc = skinny_segs(n, k, 2, a, bp, cp, ms, segs, nslab, blocks16);
    if (rc) return rc;
    (void)blocks16;
    const uint32_t kp = (uint32_t)round_up(k, BK);
    const uint32_t waves = skinny_waves(k, 2);      // 16 gate and 16 up columns a workgroup
    CM_LAUNCH("skinny_mulact_kernel", skinny_mulact_kernel<2>, dim3(ceil_div(m, 16)), dim3(64 * waves),
              skinny_lds(waves, 2), s, a, n, k, kp, nslab, segs, mj);
    return CM_OK;
}

}  // namespace
}  // namespace cm

extern "C" int cm_matmul_skinny_planes_mulact(const int16_t* a, uint32_t n, uint32_t k, const void* b_gate,
                                              const void* b_up, int16_t* c_gate, int16_t* c_up, uint32_t m,
                                              const void* params, uint32_t op, int16_t* out, void* stream) {
    using namespace cm;
    DeviceState* st;
    int rc = state(&st);
    if (rc) return rc;
    if ((op & 15) != ro::RO_MULACT || !(op & ro::F_B_EN) || (op & ro::F_P_KEEP) || ((op >> 4) & 3) != 0 ||
        ((op >> 6) & 3) != 0 || ((op >> 8) & 3) != 0)
        return fail(CM_EINVAL, "matmul: the output job must be an int16 MULACT with B enabled (op 0x%x)", op);
    if (params == nullptr || out == nullptr || c_gate == nullptr || c_up == nullptr)
        return fail(CM_EINVAL, "matmul: the MULACT output needs both products, out and a parameter block");
    if (m > ro::kNMax) return fail(CM_EINVAL, "matmul: the MULACT job's rows of %u above %u", m, ro::kNMax);
    if ((reinterpret_cast<uintptr_t>(params) & 15) || (reinterpret_cast<uintptr_t>(out) & 1) ||
        (reinterpret_cast<uintptr_t>(c_gate) & 1) || (reinterpret_cast<uintptr_t>(c_up) & 1))
        return fail(CM_EALIGN, "matmul: the MULACT operands are not aligned");
    const SkinnyMulact mj{out, static_cast<const uint8_t*>(params), (op & ro::F_P_BCAST) ? 1u : 0u, st->ro_tables};
    return skinny_mulact(a, n, k, b_gate, b_up, c_gate, c_up, m, mj, as_stream(stream));
}

extern "C" int cm_matmul_skinny_planes(const int16_t* a, uint32_t n, uint32_t k, uint32_t count,
                                       const void* const* b_planes, int16_t* const* c, const uint32_t* m,
                                       void* stream) {
    using namespace cm;
    DeviceState* st;
    int rc = state(&st);
    if (rc) return rc;
    return skinny_planes(a, n, k, count, b_planes, c, m, SkinnyAddx{}, as_stream(stream));
}

extern "C" int cm_matmul_skinny_planes_sat(const int16_t* a, uint32_t n, uint32_t k, uint32_t count,
                                           const void* const* b_planes, int16_t* const* c, const uint32_t* m,
                                           void* stream) {
    using namespace cm;
    DeviceState* st;
    int rc = state(&st);
    if (rc) return rc;
    return skinny_planes(a, n, k, count, b_planes, c, m, SkinnyAddx{}, as_stream(stream), true);
}

extern "C" int cm_matmul_skinny_planes_addx(const int16_t* a, uint32_t n, uint32_t k, const void* b_planes,
                                            int16_t* c, uint32_t m, const void* x, const void* params, uint32_t op,
                                            uint32_t bq_sh, void* out, void* stream) {
    using namespace cm;
    DeviceState* st;
    int rc = state(&st);
    if (rc) return rc;
    const uint32_t code = op & 15, ak = (op >> 4) & 3, bk = (op >> 6) & 3, ck = (op >> 8) & 3;
    if ((code != ro::RO_COPY && code != ro::RO_ADDX) || !(op & ro::F_B_EN) || (op & ro::F_P_KEEP) || ak > 1 ||
        bk != 0 || ck > 1 || bq_sh > 63)
        return fail(CM_EINVAL, "matmul: the output job must be a COPY / ADDX with B the int16 product (op 0x%x)", op);
    if (x == nullptr || out == nullptr || params == nullptr)
        return fail(CM_EINVAL, "matmul: the output job needs x, out and a parameter block");
    if ((reinterpret_cast<uintptr_t>(x) & (ak ? 3 : 1)) || (reinterpret_cast<uintptr_t>(out) & (ck ? 3 : 1)) ||
        (reinterpret_cast<uintptr_t>(params) & 15))
        return fail(CM_EALIGN, "matmul: the output job's operands are not aligned");
    const SkinnyAddx ax{static_cast<const uint8_t*>(x), static_cast<uint8_t*>(out), static_cast<const uint8_t*>(params),
                        op, bq_sh};
    return skinny_planes(a, n, k, 1, &b_planes, &c, &m, ax, as_stream(stream));
}
