// Single grid points of the attention evaluated over their true neighbors only, by one wavefront: forward, dq and dk/dv.
// Included by s2attn_kernels.hip inside namespace s2 after s2attn_h16.hpp; called at the end of the kernels of s2attn_s16.hpp and
// s2attn_m32.hpp for the columns whose result is not finite.
//
// A matrix-core tile multiplies rows a column does not see by a probability of zero, and 0 x NaN is NaN: one missing value would
// reach every column whose tile holds it.  Split operands also turn an infinity (and a magnitude above bf16's largest, 3.39e38) into NaN,
// and log2 of a negative quadrature weight is NaN.  All of these show in the sums, so a column with finite sums is right as it
// stands, and the others are evaluated again here, where an operand meets the points that see it and no other, as itself.  The check
// is one addition per accumulator register at the end of a walk; a tile without such values pays nothing else.  (Walking again over a
// staged band without such values, in the same kernel, would keep the bits of the columns that do not see them, and costs the
// walk 10 to 50 registers: a wavefront per SIMD in most forwards.)
//
// SEEN: only columns that do see such a value (or a magnitude above 2e38, or an unusual weight) are written; the others keep the tile's
// result.  For fp32 heads of 32 channels, which run on the hybrid kernels or on split products as the grid has it: what is not
// finite may reach a whole tile on both, and what stays finite has the same bits with and without it.
//
// Lane l = (j = l % 16, g = l / 16): four neighbors at a time, the lanes of a group share one neighbor's channels (j, j + 16, ...).
// Bound by the latency of the loads: about ten times slower than the tiles where everything is NaN.

// The evaluation reads the arguments of the kernel again and counts the lanes anew, so nothing is kept in registers through a walk for it
// (kept there, it cost the 16-channel forward one of its five wavefronts per SIMD), and stands behind the end of its kernel (among the
// blocks of the walk it cost the 16-channel fp32 tiles 2 %).
__device__ inline Args point_args()
{
    typedef const int __attribute__((address_space(4))) * words;
    words p = (words)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    Args a;
    static_assert(sizeof(Args) % 4 == 0, "read as 32-bit words");
#pragma unroll
    for (unsigned i = 0; i < sizeof(Args) / 4; i++) reinterpret_cast<int *>(&a)[i] = p[i];
    return a;
}
__device__ inline int point_lane()
{
    unsigned zero = 0;
    asm volatile("" : "+s"(zero));
    return (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, zero));
}

// Columns (bits 0 .. 15) in which any of the four lanes of the column says so
__device__ inline unsigned point_columns(bool any)
{
    const unsigned long long l = __ballot(any);
    return (unsigned)((l | l >> 16 | l >> 32 | l >> 48) & 0xffffu);
}
__device__ inline bool not_finite(float x) { return !(fabsf(x) < INFINITY); }
__device__ inline float point_sum(f4v x) { return (x[0] + x[1]) + (x[2] + x[3]); }

__device__ inline bool unusual(float x) { return !(fabsf(x) < 2.0e38f); }
__device__ inline bool unusual_weight(float w) { return !(w >= 0.f && w < INFINITY); }

// <x, y> over n channels, in all sixteen lanes of the group; far: an unusual value was met (the neighbor counts: in)
template <typename T> __device__ inline float point_dot(const T *x, const T *y, int n, int j, bool in, bool &far)
{
    float s = 0.f;
    for (int c = j; c < n; c += 16) {
        const float a = to_f32(x[c]), b = to_f32(y[c]);
        far |= in && (unusual(a) || unusual(b));
        s = fmaf(a, b, s);
    }
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) s += __shfl_xor(s, o);
    return s;
}

// out[c] = x[c] over the four groups' shares, channels c = j + 16 i < nc
template <typename T, int N> __device__ inline void point_store(T *out, const float (&x)[N], float scale, int nc, int j, int g)
{
#pragma unroll
    for (int i = 0; i < N; i++) {
        const float s = h16_quarter_sum(x[i]) * scale;
        if (g == 0 && j + 16 * i < nc) from_f32(out[j + 16 * i], s);
    }
}

// y of one query, channels c0 .. c0 + nc (at most 16 N) of its head, and with `stat` its softmax normaliser
template <typename T, int N, bool SEEN> __device__ inline void point_forward(const Args &a, int b, int h, int bh, int ho, int wo, int c0, int nc, bool stat, int lane)
{
    const int j = lane & 15, g = lane >> 4;
    const size_t pq = (size_t)query_point(a, b, ho, ho / a.qps) + (size_t)wo * a.qps;
    const T *q = static_cast<const T *>(a.q) + pq * a.ldq + h * a.dk_;
    float acc[N] = {}, m = NEG_BIG, Z = 0.f;
    bool far = false;
    for (int ri = a.goff[ho]; ri < a.goff[ho + 1]; ri++) {
        const Run run = a.gruns[ri];
        const float w = a.quad_w[run.pad];
        const size_t row = (size_t)key_point(a, b, run.lat, run.pad);
        for (int t0 = 0; t0 < run.len; t0 += 4) {
            const bool in = t0 + g < run.len;
            const size_t pk = row + (size_t)((run.ws + wo + t0 + (in ? g : 0)) % a.Wi) * a.kps;
            const float s = point_dot(q, static_cast<const T *>(a.k) + pk * a.ldk + h * a.dk_, a.dk_, j, in, far) * LOG2E;
            if (in) {
                far |= unusual_weight(w);
                const T *v = static_cast<const T *>(a.v) + pk * a.ldv + h * a.dv_ + c0;
                const float mn = fmaxf(m, s), corr = fast_exp2(m - mn), p = fast_exp2(s - mn) * w;
                m = mn;
                Z = fmaf(Z, corr, p);
#pragma unroll
                for (int i = 0; i < N; i++) {
                    if (j + 16 * i < nc) {
                        const float x = to_f32(v[j + 16 * i]);
                        far |= unusual(x);
                        acc[i] = fmaf(p, x, acc[i] * corr);
                    }
                }
            }
        }
    }
    if (SEEN && !__any(far)) return;
    const float mx = h16_quarter_max(m), f = fast_exp2(m - mx);
    Z = h16_quarter_sum(Z * f);
#pragma unroll
    for (int i = 0; i < N; i++) acc[i] *= f;
    point_store(static_cast<T *>(a.y) + pq * a.ldy + h * a.dv_ + c0, acc, 1.f / Z, nc, j, g);
    if (stat && a.lse && lane == 0) a.lse[((size_t)bh * a.Ho + ho) * a.Wo + wo] = mx + fast_log2(Z);
}

// dq of one query from the forward's y and lse, channels c0 .. c0 + nc of its head, and with `stat` its two statistics.  16-bit storage:
// the mean of <dy, v> is brought from <dy, y> of the rounded y to that of the probabilities, as in dq_s16_kernel.
template <typename T, int N, bool SEEN> __device__ inline void point_dq(const Args &a, int b, int h, int bh, int ho, int wo, int c0, int nc, bool stat, int lane)
{
    const int j = lane & 15, g = lane >> 4;
    const size_t pq = (size_t)query_point(a, b, ho, ho / a.qps) + (size_t)wo * a.qps, si = ((size_t)bh * a.Ho + ho) * a.Wo + wo;
    const T *q = static_cast<const T *>(a.q) + pq * a.ldq + h * a.dk_, *dy = static_cast<const T *>(a.dy) + pq * a.ldg + h * a.dv_;
    bool far = false;
    const float I = point_dot(dy, static_cast<const T *>(a.ysaved) + pq * a.ldy + h * a.dv_, a.dv_, j, true, far), lse = a.lse[si];
    far |= unusual(lse);
    constexpr bool EXACT_I = std::is_same<T, float>::value;
    float acc[N] = {}, ak[EXACT_I ? 1 : N] = {}, off = 0.f;
    for (int ri = a.goff[ho]; ri < a.goff[ho + 1]; ri++) {
        const Run run = a.gruns[ri];
        const float w = a.quad_w[run.pad];
        const size_t row = (size_t)key_point(a, b, run.lat, run.pad);
        for (int t0 = 0; t0 < run.len; t0 += 4) {
            const bool in = t0 + g < run.len;
            const size_t pk = row + (size_t)((run.ws + wo + t0 + (in ? g : 0)) % a.Wi) * a.kps;
            const T *k = static_cast<const T *>(a.k) + pk * a.ldk + h * a.dk_;
            const float s = point_dot(q, k, a.dk_, j, in, far), gv = point_dot(dy, static_cast<const T *>(a.v) + pk * a.ldv + h * a.dv_, a.dv_, j, in, far);
            if (in) {
                far |= unusual_weight(w);
                const float p = fast_exp2(fmaf(s, LOG2E, -lse)) * w, ds = p * (gv - I);
                if (!EXACT_I) off += ds;
#pragma unroll
                for (int i = 0; i < N; i++) {
                    if (j + 16 * i < nc) {
                        const float x = to_f32(k[c0 + j + 16 * i]);
                        acc[i] = fmaf(ds, x, acc[i]);
                        if (!EXACT_I) ak[EXACT_I ? 0 : i] = fmaf(p, x, ak[EXACT_I ? 0 : i]);
                    }
                }
            }
        }
    }
    if (SEEN && !__any(far)) return;
    off = h16_quarter_sum(off);
    if (!EXACT_I) {
#pragma unroll
        for (int i = 0; i < N; i++) acc[i] = fmaf(-off, ak[EXACT_I ? 0 : i], acc[i]);
    }
    point_store(static_cast<T *>(a.dq) + pq * a.lddq + h * a.dk_ + c0, acc, 1.f, nc, j, g);
    if (stat && lane == 0) a.stats[si] = make_float2(lse, I + off);
}

// dk and dv of one key, channels c0 .. c0 + nk and c0 .. c0 + nv of its head
template <typename T, int N, bool SEEN> __device__ inline void point_dkdv(const Args &a, int b, int h, int bh, int hi, int wi, int c0, int nk, int nv, int lane)
{
    const int j = lane & 15, g = lane >> 4;
    const size_t pk = (size_t)key_point(a, b, hi, hi / a.kps) + (size_t)wi * a.kps;
    const T *k = static_cast<const T *>(a.k) + pk * a.ldk + h * a.dk_, *v = static_cast<const T *>(a.v) + pk * a.ldv + h * a.dv_;
    const float w = a.quad_w[hi / a.kps];
    float dk[N] = {}, dv[N] = {};
    bool far = unusual_weight(w);
    for (int ri = a.soff[hi]; ri < a.soff[hi + 1]; ri++) {
        const Run run = a.sruns[ri]; // the key is neighbor t of query column wi - ws - t
        const size_t row = (size_t)query_point(a, b, run.lat, run.pad), srow = ((size_t)bh * a.Ho + run.lat) * a.Wo;
        for (int t0 = 0; t0 < run.len; t0 += 4) {
            const bool in = t0 + g < run.len;
            int col = (wi - run.ws - t0 - (in ? g : 0)) % a.Wo;
            col += col < 0 ? a.Wo : 0;
            const size_t pq = row + (size_t)col * a.qps;
            const T *q = static_cast<const T *>(a.q) + pq * a.ldq + h * a.dk_, *dy = static_cast<const T *>(a.dy) + pq * a.ldg + h * a.dv_;
            const float s = point_dot(q, k, a.dk_, j, in, far), gv = point_dot(dy, v, a.dv_, j, in, far);
            if (in) {
                const float2 st = a.stats[srow + col];
                far |= unusual(st.x) || unusual(st.y);
                const float p = fast_exp2(fmaf(s, LOG2E, -st.x)) * w, ds = p * (gv - st.y);
#pragma unroll
                for (int i = 0; i < N; i++) {
                    if (j + 16 * i < nv) dv[i] = fmaf(p, to_f32(dy[c0 + j + 16 * i]), dv[i]);
                    if (j + 16 * i < nk) dk[i] = fmaf(ds, to_f32(q[c0 + j + 16 * i]), dk[i]);
                }
            }
        }
    }
    if (SEEN && !__any(far)) return;
    point_store(static_cast<T *>(a.dk) + pk * a.lddk + h * a.dk_ + c0, dk, 1.f, nk, j, g);
    point_store(static_cast<T *>(a.dv) + pk * a.lddv + h * a.dv_ + c0, dv, 1.f, nv, j, g);
}
