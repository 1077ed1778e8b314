// The module's 1x1 projections on the matrix cores: NCHW activations -> NHWC q, k, v (and back), their input and weight
// gradients, and the per-head RMS norm of q and k.  (The reference runs four F.linear between two layout copies,
// attention.py:519-571.)
//
// All products are of one of two forms; "channel-major" is a [C][n] image of an NCHW tensor, "point-major" a [n][C] one of
// an NHWC tensor (n = grid points of one batch element):
//   projection   out[n, o] = sum_c X[c, n] W[o, c]   channel-major in, point-major out   (q, k, v; input gradient of the output projection)
//                out[o, n] = sum_c W[o, c] Y[n, c]   point-major in, channel-major out   (output projection; input gradient of q, k, v)
//   reduction    R[i, j]   = sum_n P[i, n] Q[n, j]   one operand of each kind            (weight gradients; bias gradients on the side)
// so no layout copy of an activation is ever made: a tile is transposed, if it has to be, on its way into LDS.
//
// Arithmetic.  v_mfma_f32_32x32x16_{bf16,f16}, fp32 accumulation.  16-bit activations (or fp32 ones under autocast) enter as
// they are (rounded once).  fp32 activations enter as three bf16 terms, x = h + m + l, each the round-to-nearest bf16 of what the
// earlier ones left (|x - h - m - l| <= 2^-25 |x|, below half an ulp of x), and a product is the six term products of at
// most second order; the three left out are below 2^-26 of the product, a quarter of the rounding an fp32 multiply makes.  The
// fp32 matrix instructions have a sixteenth of the bf16 rate (157 against 2,500 TFLOP/s), so six products cost 6/16.
//
// Weights are small and shared by every workgroup: a pack kernel lays them out once per call in the order the matrix
// instructions take them (block of 64 rows, 16 channels, term, 64 lanes x 16 bytes), so a wavefront loads its operand straight from
// L2 into registers, fully coalesced, and LDS holds activations only.

#include "s2attn_internal.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

namespace s2proj {

typedef unsigned u4v __attribute__((ext_vector_type(4)));
typedef float f4v __attribute__((ext_vector_type(4)));
typedef float f16v __attribute__((ext_vector_type(16)));
typedef float f2v __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
// rows of an activation start at any multiple of the element size (odd channel counts, odd grids); gfx950 loads vectors
// from such addresses as they are
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
typedef unsigned u4u __attribute__((ext_vector_type(4), aligned(2)));
typedef unsigned u1u __attribute__((aligned(2)));

struct bf16_t {
    unsigned short u;
};
struct f16_t {
    unsigned short u;
};

__device__ inline float up(float x) { return x; }
__device__ inline float up(bf16_t x) { return __uint_as_float((unsigned)x.u << 16); }
__device__ inline float up(f16_t x) { return (float)__builtin_bit_cast(_Float16, x.u); }
template <typename T> __device__ inline float up_lo(unsigned p);
template <typename T> __device__ inline float up_hi(unsigned p);
template <> __device__ inline float up_lo<bf16_t>(unsigned p) { return __uint_as_float(p << 16); }
template <> __device__ inline float up_hi<bf16_t>(unsigned p) { return __uint_as_float(p & 0xffff0000u); }
template <> __device__ inline float up_lo<f16_t>(unsigned p) { return (float)__builtin_bit_cast(f16x2_t, p)[0]; }
template <> __device__ inline float up_hi<f16_t>(unsigned p) { return (float)__builtin_bit_cast(f16x2_t, p)[1]; }
__device__ inline unsigned pack2(float a, float b, bf16_t)
{
    const f2v x = {a, b};
    return __builtin_bit_cast(unsigned, __builtin_convertvector(x, bf16x2_t));
}
__device__ inline unsigned pack2(float a, float b, f16_t)
{
    const f2v x = {a, b};
    return __builtin_bit_cast(unsigned, __builtin_convertvector(x, f16x2_t));
}
__device__ inline void put(float *p, float x) { *p = x; }
__device__ inline void put(bf16_t *p, float x) { p->u = (unsigned short)pack2(x, x, bf16_t{}); }
__device__ inline void put(f16_t *p, float x) { p->u = (unsigned short)pack2(x, x, f16_t{}); }

// How a product is computed: NT terms per value, KC channels (or points, in the reduction) per staged chunk.
struct Split3 { // fp32 as three bf16 terms
    static constexpr int NT = 3, KC = 32;
    static __device__ inline float round(float x) { return x; }
    static __device__ inline void convert(u4v *t, const float (&v)[8])
    {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float a = v[2 * i], b = v[2 * i + 1];
            const unsigned h = pack2(a, b, bf16_t{});
            const float ra = a - up_lo<bf16_t>(h), rb = b - up_hi<bf16_t>(h);
            const unsigned m = pack2(ra, rb, bf16_t{});
            t[0][i] = h, t[1][i] = m, t[2][i] = pack2(ra - up_lo<bf16_t>(m), rb - up_hi<bf16_t>(m), bf16_t{});
        }
    }
    static __device__ inline f16v mma1(u4v a, u4v b, f16v c)
    {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
    }
    // The five low-order products go to a sum of their own (2^-8 of the other one): the main sum is rounded once per 16 k
    // instead of six times, which measures 1.2e-7 relative at 256 channels against 2.9e-7 in one sum (fp32 GEMM: 2.0e-7).
    static constexpr int NS = 2;
    static __device__ inline void mma(const u4v *a, const u4v *b, f16v *c)
    {
        c[1] = mma1(a[2], b[0], c[1]);
        c[0] = mma1(a[0], b[0], c[0]);
        c[1] = mma1(a[0], b[2], c[1]);
        c[1] = mma1(a[1], b[1], c[1]);
        c[1] = mma1(a[1], b[0], c[1]);
        c[1] = mma1(a[0], b[1], c[1]);
    }
};
template <typename H> struct Half16 {
    static constexpr int NT = 1, KC = 64;
    static __device__ inline float round(float x) { return up_lo<H>(pack2(x, x, H{})); }
    static __device__ inline void convert(u4v *t, const float (&v)[8])
    {
#pragma unroll
        for (int i = 0; i < 4; i++) t[0][i] = pack2(v[2 * i], v[2 * i + 1], H{});
    }
};
struct MulBf16 : Half16<bf16_t> {
    static constexpr int NS = 1;
    static __device__ inline void mma(const u4v *a, const u4v *b, f16v *c)
    {
        c[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a[0]), __builtin_bit_cast(bf16x8_t, b[0]), c[0], 0, 0, 0);
    }
};
struct MulF16 : Half16<f16_t> {
    static constexpr int NS = 1;
    static __device__ inline void mma(const u4v *a, const u4v *b, f16v *c)
    {
        c[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a[0]), __builtin_bit_cast(f16x8_t, b[0]), c[0], 0, 0, 0);
    }
};

// ---- staging ------------------------------------------------------------------------------------------------------------
// A staged tile is ROWS rows (points, or channels of a reduction) of [term][KC] 16-bit values, 16 bytes of padding per row: the
// 16-byte reads of a matrix operand (lane = row, 8 consecutive k) and the 16-byte writes are free of bank conflicts at both
// pitches (208 and 144 bytes).
template <typename C> constexpr int PITCH = C::NT *C::KC * 2 + 16;

// Source whose k index is strided and whose row index is contiguous: element (k, r) at base[k * ks + r].  A lane gathers 8
// consecutive k of one row (two rows of 16-bit elements), which is what it writes to LDS: the transposition costs nothing.
// A wavefront takes slots of 64 rows (16-bit: 128, or 64 rows x 2 octets) x 8 k.
template <typename TI, typename C, int ROWS, int NWV, bool SUM> struct StageT {
    static constexpr bool WIDE = sizeof(TI) == 4;
    static constexpr int GROUPS = !WIDE && ROWS == 64 ? 2 : 1; // octets of k side by side in a wavefront
    static constexpr int LPG = 64 / GROUPS, RPS = WIDE ? 64 : 2 * LPG; // lanes per octet, rows per slot
    static constexpr int RG = ROWS / RPS, NS = RG * (C::KC / 8 / GROUPS) / NWV, PER = WIDE ? 1 : 2;
    static_assert(NS >= 1 && RG * (C::KC / 8 / GROUPS) % NWV == 0 && (RG == 1 || NWV % RG == 0), "slots do not divide evenly");
    unsigned v[NS][8], shift;
    float sum[PER];

    const TI *base;
    int64_t ks;
    int row0, rows; // first row of the tile; rows of the source
    int lane, wave;

    __device__ inline void init(int l, int w)
    {
        lane = l, wave = w;
        if (SUM) {
#pragma unroll
            for (int i = 0; i < PER; i++) sum[i] = 0.f;
        }
    }
    // the rows of a lane are the same in all its slots
    __device__ inline int row() const { return (wave % RG) * RPS + PER * (GROUPS > 1 ? lane % LPG : lane); }
    __device__ inline int octet(int i) const { return ((wave + NWV * i) / RG) * GROUPS + (GROUPS > 1 ? lane / LPG : 0); }
    // k from kend on: zeros where the sums over k are wanted (a reduction, whose other operand is zero there as well), else the last
    // value again: the weights it meets are zero
    __device__ inline void load(int k0, int kend)
    {
        const int r = row0 + row();
        if constexpr (WIDE) {
            const float *p = reinterpret_cast<const float *>(base) + min(r, rows - 1);
#pragma unroll
            for (int i = 0; i < NS; i++)
#pragma unroll
                for (int j = 0; j < 8; j++) v[i][j] = __float_as_uint(p[(int64_t)min(k0 + 8 * octet(i) + j, kend - 1) * ks]);
        } else {
            // last row of an odd count: the pair before it is loaded and shifted down when it is stored
            shift = rows >= 2 && r == rows - 1 ? 16u : 0u;
            const unsigned short *p = reinterpret_cast<const unsigned short *>(base) + min(r, max(rows - 2, 0));
            if (rows >= 2) {
#pragma unroll
                for (int i = 0; i < NS; i++)
#pragma unroll
                    for (int j = 0; j < 8; j++) v[i][j] = *reinterpret_cast<const u1u *>(p + (int64_t)min(k0 + 8 * octet(i) + j, kend - 1) * ks);
            } else {
#pragma unroll
                for (int i = 0; i < NS; i++)
#pragma unroll
                    for (int j = 0; j < 8; j++) v[i][j] = p[(int64_t)min(k0 + 8 * octet(i) + j, kend - 1) * ks];
            }
        }
        if (SUM && k0 + C::KC > kend) {
#pragma unroll
            for (int i = 0; i < NS; i++)
#pragma unroll
                for (int j = 0; j < 8; j++) v[i][j] = k0 + 8 * octet(i) + j < kend ? v[i][j] : 0u;
        }
    }
    __device__ inline void store(char *lds)
    {
        char *row_p = lds + row() * PITCH<C>;
#pragma unroll
        for (int i = 0; i < NS; i++) {
            char *p = row_p + 16 * octet(i);
            if constexpr (WIDE) {
                float f[8];
#pragma unroll
                for (int j = 0; j < 8; j++) f[j] = __uint_as_float(v[i][j]);
                if (SUM) sum[0] += ((f[0] + f[1]) + (f[2] + f[3])) + ((f[4] + f[5]) + (f[6] + f[7]));
                u4v t[C::NT];
                C::convert(t, f);
#pragma unroll
                for (int n = 0; n < C::NT; n++) *reinterpret_cast<u4v *>(p + n * 2 * C::KC) = t[n];
            } else {
                u4v a, b;
                const unsigned lo = shift ? 0x07060302u : 0x05040100u;
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    a[j] = __builtin_amdgcn_perm(v[i][2 * j + 1], v[i][2 * j], lo);
                    b[j] = __builtin_amdgcn_perm(v[i][2 * j + 1], v[i][2 * j], 0x07060302u);
                }
                if (SUM) {
#pragma unroll
                    for (int j = 0; j < 4; j++) sum[0] += up_lo<TI>(a[j]) + up_hi<TI>(a[j]), sum[PER - 1] += up_lo<TI>(b[j]) + up_hi<TI>(b[j]);
                }
                *reinterpret_cast<u4v *>(p) = a;
                *reinterpret_cast<u4v *>(p + PITCH<C>) = b;
            }
        }
    }
    // sums over k of every row: PARTS partial sums per row in LDS, part[PARTS][ROWS], to be added up by the caller
    static constexpr int PARTS = NWV / RG * GROUPS;
    __device__ inline void put_sums(float *part) const
    {
        const int g = (wave / RG) * GROUPS + (GROUPS > 1 ? lane / LPG : 0);
#pragma unroll
        for (int i = 0; i < PER; i++) part[g * ROWS + row() + i] = sum[i];
    }
};

// Source whose k index is contiguous: element (k, r) at base[r * rs + k].
template <typename TI, typename C, int ROWS, int NWV, bool SUM> struct StageD {
    static constexpr bool WIDE = sizeof(TI) == 4;
    static constexpr int OCT = C::KC / 8, RPP = 64 * NWV / OCT, NR = ROWS / RPP; // octets per row, rows per pass, passes
    static_assert(NR >= 1 && ROWS % RPP == 0, "rows do not divide evenly");
    u4v v[NR][WIDE ? 2 : 1];
    float sum[NR];

    const TI *base;
    int64_t rs;
    int row0, rows;
    int oct, r0;

    __device__ inline void init(int tid)
    {
        oct = tid % OCT, r0 = tid / OCT;
        if (SUM) {
#pragma unroll
            for (int i = 0; i < NR; i++) sum[i] = 0.f;
        }
    }
    __device__ inline void load(int k0, int kend)
    {
        const int k = k0 + 8 * oct;
        if (k0 + C::KC <= kend) {
#pragma unroll
            for (int i = 0; i < NR; i++) {
                const TI *p = base + (int64_t)min(row0 + r0 + i * RPP, rows - 1) * rs + k;
                if constexpr (WIDE) {
                    v[i][0] = __builtin_bit_cast(u4v, *reinterpret_cast<const f4u *>(p));
                    v[i][1] = __builtin_bit_cast(u4v, *reinterpret_cast<const f4u *>(p + 4));
                } else {
                    v[i][0] = *reinterpret_cast<const u4u *>(p);
                }
            }
            return;
        }
#pragma unroll
        for (int i = 0; i < NR; i++) {
            const TI *p = base + (int64_t)min(row0 + r0 + i * RPP, rows - 1) * rs + k;
            if (k + 8 <= kend) {
                if constexpr (WIDE) {
                    v[i][0] = __builtin_bit_cast(u4v, *reinterpret_cast<const f4u *>(p));
                    v[i][1] = __builtin_bit_cast(u4v, *reinterpret_cast<const f4u *>(p + 4));
                } else {
                    v[i][0] = *reinterpret_cast<const u4u *>(p);
                }
            } else {
#pragma unroll
                for (int h = 0; h < (WIDE ? 2 : 1); h++) v[i][h] = u4v{0u, 0u, 0u, 0u};
#pragma unroll
                for (int j = 0; j < 8; j++)
                    if (k + j < kend) {
                        if constexpr (WIDE)
                            v[i][j / 4][j % 4] = __float_as_uint(reinterpret_cast<const float *>(p)[j]);
                        else
                            v[i][0][j / 2] |= (unsigned)reinterpret_cast<const unsigned short *>(p)[j] << (16 * (j % 2));
                    }
            }
        }
    }
    __device__ inline void store(char *lds)
    {
#pragma unroll
        for (int i = 0; i < NR; i++) {
            u4v t[C::NT];
            if constexpr (WIDE) {
                float f[8];
#pragma unroll
                for (int j = 0; j < 8; j++) f[j] = __uint_as_float(v[i][j / 4][j % 4]);
                if (SUM) sum[i] += ((f[0] + f[1]) + (f[2] + f[3])) + ((f[4] + f[5]) + (f[6] + f[7]));
                C::convert(t, f);
            } else {
                t[0] = v[i][0];
                if (SUM) {
#pragma unroll
                    for (int j = 0; j < 4; j++) sum[i] += up_lo<TI>(t[0][j]) + up_hi<TI>(t[0][j]);
                }
            }
            char *p = lds + (r0 + i * RPP) * PITCH<C> + 16 * oct;
#pragma unroll
            for (int n = 0; n < C::NT; n++) *reinterpret_cast<u4v *>(p + n * 2 * C::KC) = t[n];
        }
    }
    static constexpr int PARTS = OCT;
    __device__ inline void put_sums(float *part) const
    {
#pragma unroll
        for (int i = 0; i < NR; i++) part[oct * ROWS + r0 + i * RPP] = sum[i];
    }
};

template <typename C> __device__ inline void read_operand(u4v (&t)[C::NT], const char *lds, int row, int octet)
{
    const char *p = lds + row * PITCH<C> + 16 * octet;
#pragma unroll
    for (int n = 0; n < C::NT; n++) t[n] = *reinterpret_cast<const u4v *>(p + n * 2 * C::KC);
}

// ---- weights in operand order ---------------------------------------------------------------------------------------------
struct PackArgs {
    s2attn_pack_job job[S2ATTN_PACK_MAX_JOBS];
};

template <typename TW, typename C> __device__ inline void pack_one(const s2attn_pack_job &j, int item)
{
    const int lane = item & 63, r = (item >> 6) & 1, f = item >> 7; // f = block * k16s + k16 of this job's own piece
    const int k16s = (j.cols + C::KC - 1) / C::KC * (C::KC / 16);
    const int nblk = (j.rows + 63) / 64;
    if (f >= nblk * k16s) return;
    const int blk = f / k16s, k16 = f % k16s;
    const int row = blk * 64 + r * 32 + (lane & 31), col = k16 * 16 + 8 * (lane >> 5);
    float v[8];
    const TW *w = reinterpret_cast<const TW *>(j.w);
#pragma unroll
    for (int e = 0; e < 8; e++) v[e] = row < j.rows && col + e < j.cols ? up(w[row * j.row_stride + (col + e) * j.col_stride]) * j.scale : 0.f;
    u4v t[C::NT];
    C::convert(t, v);
    u4v *dst = reinterpret_cast<u4v *>(j.dst) + ((int64_t)(j.first_block + blk) * j.total_k16 + j.first_k16 + k16) * (C::NT * 128) + r * 64 + lane;
#pragma unroll
    for (int n = 0; n < C::NT; n++) dst[n * 128] = t[n];
    if (j.dst_bias && k16 == 0 && lane < 32) {
        const float b = j.bias && row < j.rows ? up(reinterpret_cast<const TW *>(j.bias)[row]) * j.scale : 0.f;
        j.dst_bias[(j.first_block + blk) * 64 + r * 32 + lane] = C::round(b); // an operand like any other: of the type of the arithmetic
    }
}

template <typename C> __global__ __launch_bounds__(256) void pack_kernel(const PackArgs a)
{
    const s2attn_pack_job &j = a.job[blockIdx.y];
    const int item = blockIdx.x * 256 + threadIdx.x;
    switch (j.dtype) {
    case S2ATTN_F32: pack_one<float, C>(j, item); break;
    case S2ATTN_BF16: pack_one<bf16_t, C>(j, item); break;
    default: pack_one<f16_t, C>(j, item); break;
    }
}

// ---- projections ------------------------------------------------------------------------------------------------------------
struct ProjArgs {
    const void *src[S2ATTN_PROJ_MAX_PARTS];
    void *dst[S2ATTN_PROJ_MAX_PARTS];
    int src_c[S2ATTN_PROJ_MAX_PARTS], dst_c[S2ATTN_PROJ_MAX_PARTS];
    int chunk_end[S2ATTN_PROJ_MAX_PARTS]; // point-major sources: first chunk after part p
    int block_end[S2ATTN_PROJ_MAX_PARTS]; // point-major destinations: first 64-row block after part p
    int nchunks, nblocks;
    const void *w;
    const float *bias; // per row of the packed blocks, or null
    int64_t points;    // of one batch element
    int tiles_per_image, ntiles, otiles;
};

// A lane's 32 x 32 block of the result: lane = column, register i = row 8 (i / 4) + 4 (lane / 32) + i % 4.  `col` (this lane's column)
// is contiguous in the destination, row r starts r * rs elements further on; FULL: nothing lies outside.  16-bit results:
// neighboring lanes swap one of two rows, so that each stores two consecutive columns of one row.
template <bool FULL, typename TO> __device__ inline void store_block(TO *dst, const f16v &acc, int row0, int rows, int64_t rs, int col, int cols, int lane)
{
    if constexpr (sizeof(TO) == 4) {
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const int r = row0 + 8 * (i / 4) + i % 4;
            if (FULL || (col < cols && r < rows)) dst[(int64_t)r * rs + col] = acc[i];
        }
    } else {
        const int m = -(lane & 1), c = col + m; // all ones in odd lanes
#pragma unroll
        for (int i = 0; i < 16; i += 2) {
            // (bit selects: a conditional of two elements becomes a search through the vector)
            const int x0 = __float_as_int(acc[i]), x1 = __float_as_int(acc[i + 1]);
            const int send = (m & x0) | (~m & x1), keep = (m & x1) | (~m & x0);
            const int got = __builtin_amdgcn_update_dpp(0, send, 0xB1, 0xf, 0xf, false);
            const float lo = __int_as_float((m & got) | (~m & keep)), hi = __int_as_float((m & keep) | (~m & got));
            const int r = row0 + 8 * (i / 4) + i % 4 - m;
            TO *d = dst + (int64_t)r * rs + c;
            if (FULL || r < rows) {
                if (FULL || c + 1 < cols)
                    *reinterpret_cast<u1u *>(d) = pack2(lo, hi, TO{});
                else if (c < cols)
                    put(d, lo);
            }
        }
    }
}

// CM: channel-major source, point-major destinations; else point-major sources, one channel-major destination.
//
// A workgroup of WO x WN wavefronts makes WO blocks of 64 output channels x 32 NF WN points; a wavefront holds 64 x 32 NF
// accumulators (twice for split products).  The matrix cores bound it: per 16 channels a wavefront issues 2 NF (x 6) matrix
// instructions for NF (x 3) LDS reads and 2 (x 3) loads of packed weights from L2, which fly one step ahead and are issued
// before the next chunk's activations (memory returns in order: a weight load behind them would wait for HBM).
// Three staged chunks in LDS: chunk ch + 1 is written in the middle of chunk ch, behind the only barrier, so that the second half of
// the chunk's matrix instructions runs across it.
// DEEP (the largest 16-bit tile of a point-major source): a step is 8 matrix instructions, half as long as a trip to memory, and its
// weights are two registers per lane and block, so they fly three steps ahead and the next chunk is written in the last step.  1024
// channels, 361 x 720, batch 4: 9.5 -> 8.8 ms, 0.99 PFLOP/s.  A channel-major source (12.0 ms) gains nothing: its loads and LDS writes bound it.
// Which operand supplies the rows of the result decides what a lane holds of it: always one index that is contiguous in the
// destination per lane (32 lanes = 128 bytes of fp32), so stores are coalesced without a detour through LDS.
template <bool CM, typename TI, typename C, typename TO, int WO, int WN, int NF>
__global__ __launch_bounds__(64 * WO * WN, C::NT == 1 && WO * WN == 8 && NF == 2 ? 4 : 2) void proj_kernel(const ProjArgs a)
{
    constexpr int NWV = WO * WN, NTILE = 32 * NF * WN, KS = C::KC / 16, NT = C::NT, NBUF = 3;
    constexpr bool DEEP = !CM && NT == 1 && NF == 4;
    constexpr int WD = DEEP ? KS : 2, CS = DEEP ? KS - 1 : KS / 2; // sets of weight registers; step that writes the next chunk
    static_assert(KS % WD == 0, "the set of a step is known at compile time");
    __shared__ __attribute__((aligned(16))) char lds[NBUF][NTILE * PITCH<C>];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // workgroups are dealt round-robin to the 8 XCDs: the tiles of output channels that read the same points stay on one
    // XCD, next to each other in time, so all but the first find the activations in its L2
    const int q = blockIdx.x >> 3;
    const int tile = (q / a.otiles) * 8 + (blockIdx.x & 7), ot = q % a.otiles;
    if (tile >= a.ntiles) return;
    const int b = tile / a.tiles_per_image;
    const int n0 = (tile - b * a.tiles_per_image) * NTILE;
    const int npts = (int)a.points;
    const int wo = wave % WO, wn = wave / WO;
    const int blk = ot * WO + wo;
    const bool active = blk < a.nblocks;
    const int half = lane >> 5, c32 = lane & 31;

    f16v acc[2][NF][C::NS];
    {
        const float *bp = a.bias ? a.bias + (active ? blk : 0) * 64 : nullptr;
#pragma unroll
        for (int f = 0; f < 2; f++) {
            if constexpr (CM) {
                const float x = bp ? bp[f * 32 + c32] : 0.f;
#pragma unroll
                for (int i = 0; i < 16; i++) acc[f][0][0][i] = x;
            } else {
#pragma unroll
                for (int i = 0; i < 16; i++) acc[f][0][0][i] = bp ? bp[f * 32 + 8 * (i / 4) + 4 * half + i % 4] : 0.f;
            }
#pragma unroll
            for (int n = 1; n < NF; n++) acc[f][n][0] = acc[f][0][0];
#pragma unroll
            for (int n = 0; n < NF; n++)
#pragma unroll
                for (int u = 1; u < C::NS; u++)
#pragma unroll
                    for (int i = 0; i < 16; i++) acc[f][n][u][i] = 0.f;
        }
    }

    StageT<TI, C, NTILE, NWV, false> st;
    StageD<TI, C, NTILE, NWV, false> sd;
    if constexpr (CM) {
        st.init(lane, wave);
        st.base = reinterpret_cast<const TI *>(a.src[0]) + (int64_t)b * a.src_c[0] * a.points;
        st.ks = a.points, st.row0 = n0, st.rows = npts;
    } else {
        sd.init(threadIdx.x);
        sd.row0 = n0, sd.rows = npts;
    }
    auto fetch = [&](int ch) {
        if constexpr (CM) {
            st.load(ch * C::KC, a.src_c[0]);
        } else {
            const int p = ch < a.chunk_end[0] ? 0 : ch < a.chunk_end[1] ? 1 : 2;
            const int first = p ? a.chunk_end[p - 1] : 0;
            sd.base = reinterpret_cast<const TI *>(a.src[p]) + (int64_t)b * a.points * a.src_c[p];
            sd.rs = a.src_c[p];
            sd.load((ch - first) * C::KC, a.src_c[p]);
        }
    };
    auto commit = [&](char *buf) {
        if constexpr (CM)
            st.store(buf);
        else
            sd.store(buf);
    };

    const int steps = a.nchunks * KS;
    const u4v *wp = reinterpret_cast<const u4v *>(a.w) + (int64_t)(active ? blk : 0) * steps * (NT * 128) + lane;
    u4v w[WD][2][NT]; // [step modulo WD][rows 0..31 / 32..63][term]
    auto fetch_w = [&](int s, int set) {
        const u4v *p = wp + (int64_t)min(s, steps - 1) * (NT * 128);
#pragma unroll
        for (int n = 0; n < NT; n++)
#pragma unroll
            for (int f = 0; f < 2; f++) w[set][f][n] = p[n * 128 + f * 64];
    };

#pragma unroll
    for (int s = 0; s < WD - 1; s++) fetch_w(s, s);
    fetch(0);
    commit(lds[0]);
    __syncthreads();
    int cur = 0, next = 1;
    for (int ch = 0; ch < a.nchunks; ch++) {
        const bool more = ch + 1 < a.nchunks;
        const char *tilep = lds[cur] + (wn * NF * 32 + c32) * PITCH<C>;
#pragma unroll
        for (int s = 0; s < KS; s++) {
            fetch_w(ch * KS + s + WD - 1, (s + WD - 1) % WD);
            if (s == 0 && more) fetch(ch + 1);
            if (s == CS) {
                if (more) commit(lds[next]);
                __syncthreads();
            }
            if (active) {
#pragma unroll
                for (int n = 0; n < NF; n++) {
                    u4v x[NT];
                    read_operand<C>(x, tilep, n * 32, 2 * s + half);
#pragma unroll
                    for (int f = 0; f < 2; f++) CM ? C::mma(x, w[s % WD][f], acc[f][n]) : C::mma(w[s % WD][f], x, acc[f][n]);
                }
            }
        }
        cur = next, next = next == NBUF - 1 ? 0 : next + 1;
    }
    if (!active) return;
    if constexpr (C::NS == 2) {
#pragma unroll
        for (int f = 0; f < 2; f++)
#pragma unroll
            for (int n = 0; n < NF; n++)
#pragma unroll
                for (int i = 0; i < 16; i++) acc[f][n][0][i] += acc[f][n][1][i];
    }

    const int p = !CM ? 0 : blk < a.block_end[0] ? 0 : blk < a.block_end[1] ? 1 : 2;
    const int o0 = (blk - (p ? a.block_end[p - 1] : 0)) * 64, cd = a.dst_c[p];
    TO *dst = reinterpret_cast<TO *>(a.dst[p]) + (int64_t)b * a.points * cd;
    const int64_t rs = CM ? cd : a.points;
    const bool full = o0 + 64 <= cd && n0 + NTILE <= npts;
#pragma unroll
    for (int f = 0; f < 2; f++)
#pragma unroll
        for (int n = 0; n < NF; n++) {
            const int o = o0 + f * 32 + (CM ? c32 : 4 * half), pt = n0 + (wn * NF + n) * 32 + (CM ? 4 * half : c32);
            const int r = CM ? pt : o, c = CM ? o : pt;
            if (full)
                store_block<true>(dst, acc[f][n][0], r, CM ? npts : cd, rs, c, CM ? cd : npts, lane);
            else
                store_block<false>(dst, acc[f][n][0], r, CM ? npts : cd, rs, c, CM ? cd : npts, lane);
        }
}

// ---- reductions over the grid: weight and bias gradients ----------------------------------------------------------------------
struct GradArgs {
    const void *cm;                         // channel-major operand [B][ci][points]
    const void *pm[S2ATTN_PROJ_MAX_PARTS];  // point-major operands [B][points][cj]
    int ci, cj[S2ATTN_PROJ_MAX_PARTS];
    int tile_end[S2ATTN_PROJ_MAX_PARTS]; // first tile of rows after part p
    int col0[S2ATTN_PROJ_MAX_PARTS];     // first row of part p in the partial results
    int cj_total;
    int64_t points;
    int chunks_per_image, nchunks, slices, itiles, jtiles;
    float *part;     // [slices][cj_total][ci]
    float *part_cm;  // [slices][ci] sums over the points of the channel-major operand, or null
    float *part_pm;  // [slices][cj_total] of the point-major ones, or null
};

// R[j][i] = sum over a slice of the points of Q[n][j] P[i][n]: both operands are staged, both with the point index as k.  The
// slices fill the chip (the result alone has a few dozen tiles) and are added up by finish_kernel in a fixed order.
// WJ x WI wavefronts of (32 NJ) x (32 NI) results each.  Staging costs the vector unit 11 instructions per two fp32 values and LDS
// reads NJ + NI operands per NJ NI products, so the tile is as large as registers and LDS allow: 256 x 128 with eight
// wavefronts for split products, 256 x 256 for 16-bit ones.  Two chunks in LDS, one barrier per chunk.
template <typename TP, typename TQ, typename C, int WJ, int WI, int NJ, int NI>
__global__ __launch_bounds__(64 * WJ * WI, 2) void grad_kernel(const GradArgs a)
{
    constexpr int NWV = WJ * WI, TJ = 32 * WJ * NJ, TIL = 32 * WI * NI, KS = C::KC / 16, NT = C::NT, BUF = (TJ + TIL) * PITCH<C>;
    typedef StageT<TQ, C, TJ, NWV, true> StageQ;
    typedef StageD<TP, C, TIL, NWV, true> StageP;
    __shared__ __attribute__((aligned(16))) char lds[2 * BUF];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int tiles = a.itiles * a.jtiles;
    const int q = blockIdx.x >> 3;
    const int slice = (q / tiles) * 8 + (blockIdx.x & 7), tile = q % tiles; // all tiles of a slice on one XCD: they share its rows in L2
    if (slice >= a.slices) return;
    const int jt = tile / a.itiles, it = tile % a.itiles;
    const int p = jt < a.tile_end[0] ? 0 : jt < a.tile_end[1] ? 1 : 2;
    const int j0 = (jt - (p ? a.tile_end[p - 1] : 0)) * TJ, i0 = it * TIL;
    const int cj = a.cj[p];
    const int wj = wave % WJ, wi = wave / WJ;
    const int half = lane >> 5, c32 = lane & 31;

    StageQ sq;
    StageP sp;
    sq.init(lane, wave), sp.init(threadIdx.x);
    sq.ks = cj, sq.row0 = j0, sq.rows = cj;
    sp.rs = a.points, sp.row0 = i0, sp.rows = a.ci;
    auto fetch = [&](int ch) {
        const int b = ch / a.chunks_per_image, n0 = (ch - b * a.chunks_per_image) * C::KC;
        sq.base = reinterpret_cast<const TQ *>(a.pm[p]) + (int64_t)b * a.points * cj;
        sp.base = reinterpret_cast<const TP *>(a.cm) + (int64_t)b * a.ci * a.points;
        sq.load(n0, (int)a.points), sp.load(n0, (int)a.points);
    };
    f16v acc[NJ][NI][C::NS];
#pragma unroll
    for (int j = 0; j < NJ; j++)
#pragma unroll
        for (int i = 0; i < NI; i++)
#pragma unroll
            for (int u = 0; u < C::NS; u++)
#pragma unroll
                for (int e = 0; e < 16; e++) acc[j][i][u][e] = 0.f;

    const int ch0 = (int)((int64_t)a.nchunks * slice / a.slices), ch1 = (int)((int64_t)a.nchunks * (slice + 1) / a.slices);
    if (ch0 < ch1) fetch(ch0), sq.store(lds), sp.store(lds + TJ * PITCH<C>);
    __syncthreads();
    for (int ch = ch0; ch < ch1; ch++) {
        const char *lq = lds + ((ch - ch0) & 1) * BUF, *lp = lq + TJ * PITCH<C>;
        char *next = lds + ((ch - ch0 + 1) & 1) * BUF;
        const bool more = ch + 1 < ch1;
        if (more) fetch(ch + 1);
#pragma unroll
        for (int s = 0; s < KS; s++) {
            if (s == KS - 1 && more) sq.store(next), sp.store(next + TJ * PITCH<C>);
            u4v x[NI][NT];
#pragma unroll
            for (int i = 0; i < NI; i++) read_operand<C>(x[i], lp, (wi * NI + i) * 32 + c32, 2 * s + half);
#pragma unroll
            for (int j = 0; j < NJ; j++) {
                u4v y[NT];
                read_operand<C>(y, lq, (wj * NJ + j) * 32 + c32, 2 * s + half);
#pragma unroll
                for (int i = 0; i < NI; i++) C::mma(y, x[i], acc[j][i]);
            }
        }
        __syncthreads();
    }

    float *out = a.part + ((int64_t)slice * a.cj_total + a.col0[p]) * a.ci;
#pragma unroll
    for (int j = 0; j < NJ; j++)
#pragma unroll
        for (int i = 0; i < NI; i++) {
            const int ii = i0 + (wi * NI + i) * 32 + c32;
#pragma unroll
            for (int e = 0; e < 16; e++) {
                const int jj = j0 + (wj * NJ + j) * 32 + 8 * (e / 4) + 4 * half + e % 4;
                if (ii < a.ci && jj < cj) out[(int64_t)jj * a.ci + ii] = C::NS == 2 ? acc[j][i][0][e] + acc[j][i][C::NS - 1][e] : acc[j][i][0][e];
            }
        }
    const bool want_pm = a.part_pm && it == 0, want_cm = a.part_cm && jt == 0;
    float *part = reinterpret_cast<float *>(lds); // (the last chunk has been read: the loop ends with a barrier)
    if (want_pm) {
        sq.put_sums(part);
        __syncthreads();
        for (int r = threadIdx.x; r < TJ; r += 64 * NWV) {
            float s = 0.f;
            for (int g = 0; g < StageQ::PARTS; g++) s += part[g * TJ + r];
            if (j0 + r < cj) a.part_pm[(int64_t)slice * a.cj_total + a.col0[p] + j0 + r] = s;
        }
        __syncthreads();
    }
    if (want_cm) {
        sp.put_sums(part);
        __syncthreads();
        for (int r = threadIdx.x; r < TIL; r += 64 * NWV) {
            float s = 0.f;
            for (int g = 0; g < StageP::PARTS; g++) s += part[g * TIL + r];
            if (i0 + r < a.ci) a.part_cm[(int64_t)slice * a.ci + i0 + r] = s;
        }
    }
}

struct FinishArgs {
    s2attn_finish_job job[S2ATTN_FINISH_MAX_JOBS];
};

// out[r][c] = scale * sum over slices of part[slice][r][c]: 32 consecutive elements x 8 groups of slices per workgroup.  Memory latency
// bounds it (a layer of 64 channels: four 64 x 64 results of 768 slices): eight loads in flight per thread, added in the order of
// the slices, 41 -> 10 us there.
__global__ __launch_bounds__(256) void finish_kernel(const FinishArgs a)
{
    const s2attn_finish_job &j = a.job[blockIdx.y];
    const int64_t n = (int64_t)j.rows * j.cols;
    __shared__ float red[8][33];
    const int e = threadIdx.x & 31, g = threadIdx.x >> 5;
    for (int64_t base = (int64_t)blockIdx.x * 32; base < n; base += (int64_t)gridDim.x * 32) {
        const int64_t at = base + e;
        float s = 0.f;
        if (at < n) {
            const float *p = j.part + at;
            int k = g;
            for (; k + 56 < j.slices; k += 64) {
                float x[8];
#pragma unroll
                for (int i = 0; i < 8; i++) x[i] = p[(int64_t)(k + 8 * i) * j.slice_stride];
#pragma unroll
                for (int i = 0; i < 8; i++) s += x[i];
            }
            for (; k < j.slices; k += 8) s += p[(int64_t)k * j.slice_stride];
        }
        red[g][e] = s;
        __syncthreads();
        if (g == 0 && at < n) {
            float t = 0.f;
#pragma unroll
            for (int k = 0; k < 8; k++) t += red[k][e];
            t *= j.scale;
            const int64_t r = at / j.cols, c = at - r * j.cols, o = r * j.row_stride + c * j.col_stride;
            switch (j.dtype) {
            case S2ATTN_F32: reinterpret_cast<float *>(j.out)[o] = t; break;
            case S2ATTN_BF16: put(reinterpret_cast<bf16_t *>(j.out) + o, t); break;
            default: put(reinterpret_cast<f16_t *>(j.out) + o, t); break;
            }
        }
        __syncthreads();
    }
}

// ---- RMS norm of q and k over the channels of a head -----------------------------------------------------------------------
// G lanes per (point, head), each with NV pieces of V channels; 256 / G rows per pass of a workgroup.
struct NormArgs {
    const void *x[2];
    void *y[2];          // forward: the normed tensor; backward: gradient of it, replaced by the gradient of x
    const void *gain[2]; // w of the gain 1 + w
    float mult[2];
    float *dgain[2]; // backward: [blocks][d] partial sums
    int64_t rows[2];
    int d, gain_dtype;
    float eps;
};

template <typename T, int V> struct Piece;
template <> struct Piece<float, 4> {
    static __device__ inline void load(float (&f)[4], const float *p)
    {
        const f4u r = *reinterpret_cast<const f4u *>(p);
#pragma unroll
        for (int i = 0; i < 4; i++) f[i] = r[i];
    }
    static __device__ inline void store(float *p, const float (&f)[4]) { *reinterpret_cast<f4u *>(p) = f4u{f[0], f[1], f[2], f[3]}; }
};
typedef unsigned u2u __attribute__((ext_vector_type(2), aligned(2)));
template <typename T> struct Piece<T, 4> {
    static __device__ inline void load(float (&f)[4], const T *p)
    {
        const u2u r = *reinterpret_cast<const u2u *>(p);
        f[0] = up_lo<T>(r[0]), f[1] = up_hi<T>(r[0]), f[2] = up_lo<T>(r[1]), f[3] = up_hi<T>(r[1]);
    }
    static __device__ inline void store(T *p, const float (&f)[4]) { *reinterpret_cast<u2u *>(p) = u2u{pack2(f[0], f[1], T{}), pack2(f[2], f[3], T{})}; }
};
template <typename T> struct Piece<T, 1> {
    static __device__ inline void load(float (&f)[1], const T *p) { f[0] = up(*p); }
    static __device__ inline void store(T *p, const float (&f)[1]) { put(p, f[0]); }
};
__device__ inline float load_as(const void *p, int64_t i, int dtype)
{
    switch (dtype) {
    case S2ATTN_F32: return reinterpret_cast<const float *>(p)[i];
    case S2ATTN_BF16: return up(reinterpret_cast<const bf16_t *>(p)[i]);
    default: return up(reinterpret_cast<const f16_t *>(p)[i]);
    }
}
template <int G> __device__ inline float sum_over(float x)
{
#pragma unroll
    for (int o = 1; o < G; o <<= 1) x += __shfl_xor(x, o);
    return x;
}

template <typename T, int V, int NV, int G, bool BWD> __global__ __launch_bounds__(256) void norm_kernel(const NormArgs a)
{
    __shared__ float red[BWD ? 256 * V * NV : 1];
    const int t = blockIdx.y;
    const int g = threadIdx.x % G, r0 = threadIdx.x / G;
    float gain[NV][V], dg[NV][V];
#pragma unroll
    for (int n = 0; n < NV; n++)
#pragma unroll
        for (int v = 0; v < V; v++) {
            const int c = (n * G + g) * V + v;
            gain[n][v] = c < a.d ? (1.f + load_as(a.gain[t], c, a.gain_dtype)) * a.mult[t] : 0.f;
            dg[n][v] = 0.f;
        }
    const float inv = 1.f / (float)a.d;
    for (int64_t r = (int64_t)blockIdx.x * (256 / G) + r0; r < a.rows[t]; r += (int64_t)gridDim.x * (256 / G)) {
        const T *xp = reinterpret_cast<const T *>(a.x[t]) + r * a.d;
        T *yp = reinterpret_cast<T *>(a.y[t]) + r * a.d;
        float x[NV][V], y[NV][V];
        float ss = 0.f, sx = 0.f;
#pragma unroll
        for (int n = 0; n < NV; n++) {
            const int c = (n * G + g) * V;
#pragma unroll
            for (int v = 0; v < V; v++) x[n][v] = y[n][v] = 0.f;
            if (c < a.d) {
                Piece<T, V>::load(x[n], xp + c);
                if (BWD) Piece<T, V>::load(y[n], yp + c);
            }
#pragma unroll
            for (int v = 0; v < V; v++) {
                ss = fmaf(x[n][v], x[n][v], ss);
                if (BWD) sx = fmaf(gain[n][v] * y[n][v], x[n][v], sx);
            }
        }
        ss = sum_over<G>(ss);
        const float rstd = rsqrtf(fmaf(ss, inv, a.eps));
        if (BWD) sx = sum_over<G>(sx) * inv * rstd * rstd; // mean of (gain dy xhat), times rstd
#pragma unroll
        for (int n = 0; n < NV; n++) {
            const int c = (n * G + g) * V;
            float o[V];
#pragma unroll
            for (int v = 0; v < V; v++) {
                if (BWD) {
                    dg[n][v] = fmaf(y[n][v], x[n][v] * rstd, dg[n][v]);
                    o[v] = rstd * (gain[n][v] * y[n][v] - x[n][v] * sx);
                } else {
                    o[v] = x[n][v] * rstd * gain[n][v];
                }
            }
            if (c < a.d) Piece<T, V>::store(yp + c, o);
        }
    }
    if constexpr (BWD) {
#pragma unroll
        for (int n = 0; n < NV; n++)
#pragma unroll
            for (int v = 0; v < V; v++) red[r0 * (G * V * NV) + (n * G + g) * V + v] = dg[n][v];
        __syncthreads();
        for (int c = threadIdx.x; c < a.d; c += 256) {
            float s = 0.f;
            for (int r = 0; r < 256 / G; r++) s += red[r * (G * V * NV) + c];
            a.dgain[t][(int64_t)blockIdx.x * a.d + c] = s;
        }
    }
}

// ---- launches ---------------------------------------------------------------------------------------------------------------
int launched(const char *what)
{
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? S2ATTN_OK : s2attn_fail(S2ATTN_E_LAUNCH, "%s: %s", what, hipGetErrorString(e));
}

int blocks_of(int c) { return (c + 63) / 64; }

template <bool CM, typename TI, typename C, typename TO, int WO, int WN, int NF> int launch_tile(ProjArgs &a, int batch, hipStream_t s)
{
    a.tiles_per_image = (int)((a.points + 32 * NF * WN - 1) / (32 * NF * WN)), a.ntiles = batch * a.tiles_per_image;
    a.otiles = (a.nblocks + WO - 1) / WO;
    const dim3 grid((unsigned)(((int64_t)a.ntiles + 7) / 8 * 8 * a.otiles));
    proj_kernel<CM, TI, C, TO, WO, WN, NF><<<grid, 64 * WO * WN, 0, s>>>(a);
    return launched("projection");
}

template <bool CM, typename TI, typename C, typename TO> int launch_proj(ProjArgs &a, int batch, hipStream_t s)
{
    // four blocks of output channels per workgroup reuse a staged chunk most; fewer where the layer has no more or where the
    // grid would leave most of the chip idle
    const int64_t tiles = batch * ((a.points + 127) / 128);
    int wo = a.nblocks >= 3 ? 4 : a.nblocks;
    // 16-bit products: the packed weights come through the vector L1 (64 bytes per clock), which a wavefront's 64 x 64 results use
    // up; 64 x 128 halve that.  A channel-major fp32 source of few channels is the exception: its workgroups are over after a few trips to
    // memory, and two of 64 x 64 per CU overlap theirs (256 channels, 721 x 1440: 1097 -> 1043 .. 1082 us; 192, 181 x 360, batch 2: 106 -> 93;
    // a point-major 16-bit source of 256: 338 against 290)
    constexpr bool LATENCY = CM && sizeof(TI) == 4;
    if constexpr (C::NT == 1)
        if (wo == 4 && !(LATENCY && a.nchunks <= 4) && tiles / 2 * ((a.nblocks + 3) / 4) >= 512) return launch_tile<CM, TI, C, TO, 4, 2, 4>(a, batch, s);
    while (wo > 1 && tiles * ((a.nblocks + wo - 1) / wo) < 256) wo >>= 1;
    switch (wo) {
    case 4: return launch_tile<CM, TI, C, TO, 4, 2, 2>(a, batch, s);
    case 2: return launch_tile<CM, TI, C, TO, 2, 2, 2>(a, batch, s);
    default: return launch_tile<CM, TI, C, TO, 1, 4, 1>(a, batch, s);
    }
}

template <bool CM> int dispatch_proj(ProjArgs &a, const s2attn_proj *p, hipStream_t s)
{
    const int key = (p->compute * 3 + p->src_dtype) * 3 + p->dst_dtype;
    switch (key) {
    case (S2ATTN_F32 * 3 + S2ATTN_F32) * 3 + S2ATTN_F32: return launch_proj<CM, float, Split3, float>(a, p->batch, s);
    case (S2ATTN_BF16 * 3 + S2ATTN_BF16) * 3 + S2ATTN_BF16: return launch_proj<CM, bf16_t, MulBf16, bf16_t>(a, p->batch, s);
    case (S2ATTN_F16 * 3 + S2ATTN_F16) * 3 + S2ATTN_F16: return launch_proj<CM, f16_t, MulF16, f16_t>(a, p->batch, s);
    }
    if constexpr (CM) { // fp32 activations under autocast: rounded as they are staged
        if (key == (S2ATTN_BF16 * 3 + S2ATTN_F32) * 3 + S2ATTN_BF16) return launch_proj<CM, float, MulBf16, bf16_t>(a, p->batch, s);
        if (key == (S2ATTN_F16 * 3 + S2ATTN_F32) * 3 + S2ATTN_F16) return launch_proj<CM, float, MulF16, f16_t>(a, p->batch, s);
    } else { // and their gradient
        if (key == (S2ATTN_BF16 * 3 + S2ATTN_BF16) * 3 + S2ATTN_F32) return launch_proj<CM, bf16_t, MulBf16, float>(a, p->batch, s);
        if (key == (S2ATTN_F16 * 3 + S2ATTN_F16) * 3 + S2ATTN_F32) return launch_proj<CM, f16_t, MulF16, float>(a, p->batch, s);
    }
    return s2attn_fail(S2ATTN_E_UNSUPPORTED, "projection: no kernel for source %d, result %d, arithmetic %d", p->src_dtype, p->dst_dtype, p->compute);
}

int chunk_of(int compute) { return compute == S2ATTN_F32 ? Split3::KC : MulBf16::KC; }

int check_proj(const s2attn_proj *p, bool cm)
{
    if (!p) return s2attn_fail(S2ATTN_E_INVALID, "null projection");
    if (p->batch < 1 || p->points < 1 || p->points > INT32_MAX - 256) return s2attn_fail(S2ATTN_E_INVALID, "projection: bad extents");
    if (p->nsrc < 1 || p->nsrc > S2ATTN_PROJ_MAX_PARTS || p->ndst < 1 || p->ndst > S2ATTN_PROJ_MAX_PARTS || (cm ? p->nsrc : p->ndst) != 1)
        return s2attn_fail(S2ATTN_E_INVALID, "projection: bad number of parts");
    for (int i = 0; i < p->nsrc; i++)
        if (!p->src[i] || p->src_channels[i] < 1) return s2attn_fail(S2ATTN_E_INVALID, "projection: null or empty source");
    for (int i = 0; i < p->ndst; i++)
        if (!p->dst[i] || p->dst_channels[i] < 1) return s2attn_fail(S2ATTN_E_INVALID, "projection: null or empty destination");
    if (!p->packed) return s2attn_fail(S2ATTN_E_INVALID, "projection: null weights");
    for (int d : {p->src_dtype, p->dst_dtype, p->compute})
        if (d != S2ATTN_F32 && d != S2ATTN_BF16 && d != S2ATTN_F16) return s2attn_fail(S2ATTN_E_INVALID, "projection: unknown dtype %d", d);
    if ((int64_t)p->batch * ((p->points + 127) / 128) > (1 << 24)) return s2attn_fail(S2ATTN_E_UNSUPPORTED, "projection: too many points");
    return S2ATTN_OK;
}

template <bool CM> int run_proj(const s2attn_proj *p, void *stream)
{
    const int rc = check_proj(p, CM);
    if (rc != S2ATTN_OK) return rc;
    ProjArgs a = {};
    const int kc = chunk_of(p->compute);
    int ch = 0, bl = 0;
    for (int i = 0; i < S2ATTN_PROJ_MAX_PARTS; i++) {
        if (i < p->nsrc) a.src[i] = p->src[i], a.src_c[i] = p->src_channels[i], ch += (p->src_channels[i] + kc - 1) / kc;
        if (i < p->ndst) a.dst[i] = p->dst[i], a.dst_c[i] = p->dst_channels[i], bl += blocks_of(p->dst_channels[i]);
        a.chunk_end[i] = ch, a.block_end[i] = bl;
    }
    a.nchunks = ch, a.nblocks = bl, a.w = p->packed, a.bias = p->bias, a.points = p->points;
    return dispatch_proj<CM>(a, p, (hipStream_t)stream);
}

// Tiles of the weight gradient, smallest first: results (j x i), wavefronts and workgroups of it that a CU holds.
struct GradTile {
    int tj, ti, per_cu;
};
constexpr GradTile GRAD_TILES[3][3] = {{{64, 64, 3}, {128, 128, 1}, {256, 128, 1}},  // split fp32
                                       {{64, 64, 4}, {128, 128, 2}, {256, 256, 1}},  // 16-bit
                                       {{64, 64, 4}, {128, 128, 2}, {256, 128, 1}}}; // 16-bit, one operand stored in fp32
const GradTile *grad_tiles(const s2attn_grad *g) { return GRAD_TILES[g->compute == S2ATTN_F32 ? 0 : g->cm_dtype == S2ATTN_F32 ? 2 : 1]; }

template <typename TP, typename TQ, typename C> int launch_grad(GradArgs &a, int tile, hipStream_t s)
{
    const dim3 grid((unsigned)((a.slices + 7) / 8 * 8 * a.itiles * a.jtiles));
    constexpr int NI = sizeof(TP) == 4 ? 2 : 4;
    switch (tile) {
    case 0: grad_kernel<TP, TQ, C, 2, 2, 1, 1><<<grid, 256, 0, s>>>(a); break;
    case 1: grad_kernel<TP, TQ, C, 2, 4, 2, 1><<<grid, 512, 0, s>>>(a); break;
    default: grad_kernel<TP, TQ, C, 4, 2, 2, NI><<<grid, 512, 0, s>>>(a); break;
    }
    return launched("weight gradient");
}

struct GradTiling {
    int tile, itiles, jtiles, slices, nchunks, chunks_per_image, cj_total;
};

GradTiling grad_tiling(const s2attn_grad *g)
{
    const int kc = chunk_of(g->compute);
    GradTiling best = {};
    double best_cost = 0;
    for (int k = 0; k < 3; k++) {
        const GradTile &tl = grad_tiles(g)[k];
        GradTiling t = {};
        t.tile = k, t.itiles = (g->cm_channels + tl.ti - 1) / tl.ti;
        for (int i = 0; i < g->npm; i++) t.jtiles += (g->pm_channels[i] + tl.tj - 1) / tl.tj, t.cj_total += g->pm_channels[i];
        t.chunks_per_image = (int)((g->points + kc - 1) / kc);
        t.nchunks = g->batch * t.chunks_per_image;
        // A slice costs a pass over the result, so no more of them than fill the 32 CUs of every XCD a whole number of times
        // (rounds); at least four chunks each.
        const int tiles = t.itiles * t.jtiles, slots = 32 * tl.per_cu;
        const int most = std::max(1, t.nchunks / 32);
        int per_xcd = 1;
        double fill = 0;
        for (int s = 1; s <= std::min(most, std::max(1, 3 * slots / tiles)); s++) {
            const int rounds = (s * tiles + slots - 1) / slots;
            const double f = (double)(s * tiles) / (rounds * slots) - 0.01 * rounds;
            if (f > fill) fill = f, per_xcd = s;
        }
        t.slices = t.nchunks < 32 ? std::max(1, t.nchunks / 4) : 8 * per_xcd;
        // time of a tile's chunk: matrix instructions against staging (both per result tile); the rest of a ragged tile is lost
        const double work = (double)tl.tj * tl.ti + (g->compute == S2ATTN_F32 ? 24.0 : 40.0) * (tl.tj + tl.ti);
        const double cost = work * tiles / std::max(0.05, std::min(1.0, (double)t.slices * tiles / (256.0 * tl.per_cu)));
        if (k == 0 || cost < best_cost) best = t, best_cost = cost;
    }
    return best;
}

int check_grad(const s2attn_grad *g)
{
    if (!g || g->batch < 1 || g->points < 1 || g->points > INT32_MAX - 256 || g->npm < 1 || g->npm > S2ATTN_PROJ_MAX_PARTS || g->cm_channels < 1)
        return s2attn_fail(S2ATTN_E_INVALID, "weight gradient: bad extents");
    for (int i = 0; i < g->npm; i++)
        if (g->pm_channels[i] < 1) return s2attn_fail(S2ATTN_E_INVALID, "weight gradient: empty operand");
    for (int d : {g->cm_dtype, g->pm_dtype, g->compute})
        if (d != S2ATTN_F32 && d != S2ATTN_BF16 && d != S2ATTN_F16) return s2attn_fail(S2ATTN_E_INVALID, "weight gradient: unknown dtype %d", d);
    if ((int64_t)g->batch * ((g->points + 31) / 32) > (1 << 26)) return s2attn_fail(S2ATTN_E_UNSUPPORTED, "weight gradient: too many points");
    return S2ATTN_OK;
}

template <typename T, bool BWD> int launch_norm(const NormArgs &a, int blocks, int ntensors, hipStream_t s)
{
    const dim3 grid(blocks, ntensors);
    if (a.d % 4 == 0) {
        if (a.d <= 16)
            norm_kernel<T, 4, 1, 4, BWD><<<grid, 256, 0, s>>>(a);
        else if (a.d <= 32)
            norm_kernel<T, 4, 1, 8, BWD><<<grid, 256, 0, s>>>(a);
        else if (a.d <= 64)
            norm_kernel<T, 4, 1, 16, BWD><<<grid, 256, 0, s>>>(a);
        else if (a.d <= 128)
            norm_kernel<T, 4, 1, 32, BWD><<<grid, 256, 0, s>>>(a);
        else
            norm_kernel<T, 4, 2, 64, BWD><<<grid, 256, 0, s>>>(a);
    } else if (a.d <= 16) {
        norm_kernel<T, 1, 1, 16, BWD><<<grid, 256, 0, s>>>(a);
    } else if (a.d <= 128) {
        norm_kernel<T, 1, 2, 64, BWD><<<grid, 256, 0, s>>>(a);
    } else {
        norm_kernel<T, 1, 8, 64, BWD><<<grid, 256, 0, s>>>(a);
    }
    return launched("RMS norm");
}

template <bool BWD> int run_norm(const s2attn_norm *n, void *stream)
{
    if (!n || n->ntensors < 1 || n->ntensors > 2 || n->head_channels < 1) return s2attn_fail(S2ATTN_E_INVALID, "RMS norm: bad arguments");
    if (n->head_channels > 512) return s2attn_fail(S2ATTN_E_UNSUPPORTED, "RMS norm: heads of more than 512 channels");
    if (n->blocks < 1 || n->blocks > 65535) return s2attn_fail(S2ATTN_E_INVALID, "RMS norm: bad grid");
    NormArgs a = {};
    for (int i = 0; i < n->ntensors; i++) {
        if (!n->x[i] || !n->y[i] || !n->gain[i] || (BWD && !n->dgain[i])) return s2attn_fail(S2ATTN_E_INVALID, "null tensor pointer");
        a.x[i] = n->x[i], a.y[i] = n->y[i], a.gain[i] = n->gain[i], a.mult[i] = n->mult[i], a.dgain[i] = n->dgain[i], a.rows[i] = n->rows[i];
    }
    a.d = n->head_channels, a.gain_dtype = n->gain_dtype, a.eps = n->eps;
    switch (n->dtype) {
    case S2ATTN_F32: return launch_norm<float, BWD>(a, n->blocks, n->ntensors, (hipStream_t)stream);
    case S2ATTN_BF16: return launch_norm<bf16_t, BWD>(a, n->blocks, n->ntensors, (hipStream_t)stream);
    case S2ATTN_F16: return launch_norm<f16_t, BWD>(a, n->blocks, n->ntensors, (hipStream_t)stream);
    }
    return s2attn_fail(S2ATTN_E_INVALID, "RMS norm: unknown dtype %d", n->dtype);
}

} // namespace s2proj

using namespace s2proj;

extern "C" int s2attn_pack_k16(int cols, int compute)
{
    if (cols < 1) return s2attn_fail(S2ATTN_E_INVALID, "packed weights: bad column count");
    const int kc = chunk_of(compute);
    return (cols + kc - 1) / kc * (kc / 16);
}

extern "C" int64_t s2attn_pack_bytes(int blocks, int k16, int compute)
{
    if (blocks < 1 || k16 < 1) return s2attn_fail(S2ATTN_E_INVALID, "packed weights: bad extents");
    return (int64_t)blocks * k16 * (compute == S2ATTN_F32 ? 3 : 1) * 2048;
}

extern "C" int s2attn_pack_weights(const s2attn_pack_job *jobs, int njobs, int compute, void *stream)
{
    if (!jobs || njobs < 1 || njobs > S2ATTN_PACK_MAX_JOBS) return s2attn_fail(S2ATTN_E_INVALID, "packed weights: bad number of jobs");
    PackArgs a = {};
    int64_t most = 0;
    for (int i = 0; i < njobs; i++) {
        const s2attn_pack_job &j = jobs[i];
        if (!j.w || !j.dst || j.rows < 1 || j.cols < 1) return s2attn_fail(S2ATTN_E_INVALID, "packed weights: null or empty matrix");
        if (j.dtype != S2ATTN_F32 && j.dtype != S2ATTN_BF16 && j.dtype != S2ATTN_F16) return s2attn_fail(S2ATTN_E_INVALID, "packed weights: unknown dtype %d", j.dtype);
        if (j.first_k16 + s2attn_pack_k16(j.cols, compute) > j.total_k16) return s2attn_fail(S2ATTN_E_INVALID, "packed weights: columns do not fit");
        a.job[i] = j;
        most = std::max(most, (int64_t)blocks_of(j.rows) * s2attn_pack_k16(j.cols, compute) * 128);
    }
    const dim3 grid((unsigned)((most + 255) / 256), njobs);
    switch (compute) {
    case S2ATTN_F32: pack_kernel<Split3><<<grid, 256, 0, (hipStream_t)stream>>>(a); break;
    case S2ATTN_BF16: pack_kernel<MulBf16><<<grid, 256, 0, (hipStream_t)stream>>>(a); break;
    case S2ATTN_F16: pack_kernel<MulF16><<<grid, 256, 0, (hipStream_t)stream>>>(a); break;
    default: return s2attn_fail(S2ATTN_E_INVALID, "packed weights: unknown arithmetic %d", compute);
    }
    return launched("packed weights");
}

extern "C" int s2attn_proj_nchw_to_nhwc(const s2attn_proj *p, void *stream) { return run_proj<true>(p, stream); }
extern "C" int s2attn_proj_nhwc_to_nchw(const s2attn_proj *p, void *stream) { return run_proj<false>(p, stream); }

extern "C" int s2attn_grad_slices(const s2attn_grad *g)
{
    const int rc = check_grad(g);
    return rc != S2ATTN_OK ? rc : grad_tiling(g).slices;
}

extern "C" int s2attn_grad_partials(const s2attn_grad *g, void *stream)
{
    const int rc = check_grad(g);
    if (rc != S2ATTN_OK) return rc;
    if (!g->cm || !g->part) return s2attn_fail(S2ATTN_E_INVALID, "null tensor pointer");
    const GradTiling t = grad_tiling(g);
    const GradTile &tl = grad_tiles(g)[t.tile];
    GradArgs a = {};
    a.cm = g->cm, a.ci = g->cm_channels, a.points = g->points;
    int tiles = 0, cols = 0;
    for (int i = 0; i < S2ATTN_PROJ_MAX_PARTS; i++) {
        a.col0[i] = cols;
        if (i < g->npm) {
            if (!g->pm[i]) return s2attn_fail(S2ATTN_E_INVALID, "null tensor pointer");
            a.pm[i] = g->pm[i], a.cj[i] = g->pm_channels[i];
            tiles += (g->pm_channels[i] + tl.tj - 1) / tl.tj, cols += g->pm_channels[i];
        }
        a.tile_end[i] = tiles;
    }
    a.cj_total = t.cj_total, a.chunks_per_image = t.chunks_per_image, a.nchunks = t.nchunks, a.slices = t.slices;
    a.itiles = t.itiles, a.jtiles = t.jtiles;
    a.part = g->part, a.part_cm = g->part_cm, a.part_pm = g->part_pm;
    hipStream_t s = (hipStream_t)stream;
    switch ((g->compute * 3 + g->cm_dtype) * 3 + g->pm_dtype) {
    case (S2ATTN_F32 * 3 + S2ATTN_F32) * 3 + S2ATTN_F32: return launch_grad<float, float, Split3>(a, t.tile, s);
    case (S2ATTN_BF16 * 3 + S2ATTN_BF16) * 3 + S2ATTN_BF16: return launch_grad<bf16_t, bf16_t, MulBf16>(a, t.tile, s);
    case (S2ATTN_F16 * 3 + S2ATTN_F16) * 3 + S2ATTN_F16: return launch_grad<f16_t, f16_t, MulF16>(a, t.tile, s);
    case (S2ATTN_BF16 * 3 + S2ATTN_F32) * 3 + S2ATTN_BF16: return launch_grad<float, bf16_t, MulBf16>(a, t.tile, s);
    case (S2ATTN_F16 * 3 + S2ATTN_F32) * 3 + S2ATTN_F16: return launch_grad<float, f16_t, MulF16>(a, t.tile, s);
    }
    return s2attn_fail(S2ATTN_E_UNSUPPORTED, "weight gradient: no kernel for operands %d, %d, arithmetic %d", g->cm_dtype, g->pm_dtype, g->compute);
}

extern "C" int s2attn_finish(const s2attn_finish_job *jobs, int njobs, void *stream)
{
    if (!jobs || njobs < 1 || njobs > S2ATTN_FINISH_MAX_JOBS) return s2attn_fail(S2ATTN_E_INVALID, "sums of slices: bad number of jobs");
    FinishArgs a = {};
    int64_t most = 1;
    for (int i = 0; i < njobs; i++) {
        const s2attn_finish_job &j = jobs[i];
        if (!j.part || !j.out || j.rows < 1 || j.cols < 1 || j.slices < 1) return s2attn_fail(S2ATTN_E_INVALID, "sums of slices: null or empty job");
        if (j.dtype != S2ATTN_F32 && j.dtype != S2ATTN_BF16 && j.dtype != S2ATTN_F16) return s2attn_fail(S2ATTN_E_INVALID, "sums of slices: unknown dtype %d", j.dtype);
        a.job[i] = j;
        most = std::max(most, (int64_t)j.rows * j.cols);
    }
    const dim3 grid((unsigned)std::min<int64_t>((most + 31) / 32, 4096), njobs);
    finish_kernel<<<grid, 256, 0, (hipStream_t)stream>>>(a);
    return launched("sums of slices");
}

extern "C" int s2attn_head_norm(const s2attn_norm *n, void *stream) { return run_norm<false>(n, stream); }
extern "C" int s2attn_head_norm_backward(const s2attn_norm *n, void *stream) { return run_norm<true>(n, stream); }
