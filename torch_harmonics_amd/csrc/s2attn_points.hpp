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
// A column ends as soon as all it will write is NaN, which is what the tile has written: its own q (k) or its statistics, a neighbor's
// score, or by now every sum.  Bound by the latency of the loads.  Training step at 360 x 720, one head of 64, radius 0.03: 1.6 ms,
// 2.2 with NaN on 100 of the latitudes, 3.0 with NaN everywhere (63 without ending early).
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
__device__ inline bool is_nan(float x) { return x != x; }

// over the sixteen lanes of a group, in all of them
__device__ inline float point_lanes_sum(float x)
{
    x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x128, 0xf, 0xf, false)); // row_ror:8
    x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x124, 0xf, 0xf, false));
    x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x122, 0xf, 0xf, false));
    x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x121, 0xf, 0xf, false));
    return x;
}
// Is every channel NaN in one of the groups?  (each lane: are its own?)
__device__ inline bool point_all(bool mine)
{
    const unsigned long long l = __ballot(mine);
    return (l & 0xffffu) == 0xffffu || (l >> 16 & 0xffffu) == 0xffffu || (l >> 32 & 0xffffu) == 0xffffu || l >> 48 == 0xffffu;
}
template <int N> __device__ inline bool point_nan(const float (&x)[N], int n, int j)
{
    bool all = true;
#pragma unroll
    for (int i = 0; i < N; i++) all &= is_nan(x[i]) || j + 16 * i >= n;
    return all;
}

// channels j, j + 16, ... of a grid point's vector of n channels
template <typename T, int N> struct PointRow {
    float x[N];
    __device__ inline void load(const T *p, int n, int j)
    {
#pragma unroll
        for (int i = 0; i < N; i++) x[i] = j + 16 * i < n ? to_f32(p[j + 16 * i]) : 0.f;
    }
    __device__ inline float dot(const PointRow &o) const
    {
        float s = 0.f;
#pragma unroll
        for (int i = 0; i < N; i++) s = fmaf(x[i], o.x[i], s);
        return point_lanes_sum(s);
    }
    __device__ inline bool far() const
    {
        bool f = false;
#pragma unroll
        for (int i = 0; i < N; i++) f |= unusual(x[i]);
        return f;
    }
};

// out[c] = x[c] over the four groups' shares, channels c = j + 16 i < nc
template <typename T, int N> __device__ inline void point_store(T *out, const float (&x)[N], float scale, int nc, int j, int g)
{
#pragma unroll
    for (int i = 0; i < N; i++) {
        const float s = h16_quarter_sum(x[i]) * scale;
        if (g == 0 && j + 16 * i < nc) from_f32(out[j + 16 * i], s);
    }
}

// y of one query, channels c0 .. c0 + nc (at most 16 N) of its head's (at most 16 A), and with `stat` its softmax normaliser
template <typename T, int N, int A, bool SEEN> __device__ inline void point_forward(const Args &a, int b, int h, int bh, int ho, int wo, int c0, int nc, bool stat, int lane)
{
    const int j = lane & 15, g = lane >> 4;
    const size_t pq = (size_t)query_point(a, b, ho, ho / a.qps) + (size_t)wo * a.qps;
    PointRow<T, A> q, k;
    PointRow<T, N> v;
    q.load(static_cast<const T *>(a.q) + pq * a.ldq + h * a.dk_, a.dk_, j);
    float acc[N] = {}, m = NEG_BIG, Z = 0.f;
    bool far = q.far();
    if (is_nan(q.dot(q))) return;
    for (int ri = a.goff[ho]; ri < a.goff[ho + 1]; ri++) {
        const Run run = a.gruns[ri];
        const float w = a.quad_w[run.pad];
        const size_t row = (size_t)key_point(a, b, run.lat, run.pad);
        for (int t0 = 0; t0 < run.len; t0 += 4) {
            const bool in = t0 + g < run.len;
            const size_t pk = row + (size_t)((run.ws + wo + t0 + (in ? g : 0)) % a.Wi) * a.kps;
            k.load(static_cast<const T *>(a.k) + pk * a.ldk + h * a.dk_, a.dk_, j);
            v.load(static_cast<const T *>(a.v) + pk * a.ldv + h * a.dv_ + c0, nc, j);
            const float s = q.dot(k) * LOG2E;
            if (in) {
                far |= k.far() || v.far() || unusual_weight(w);
                const float mn = fmaxf(m, s), corr = fast_exp2(m - mn), p = fast_exp2(s - mn) * w;
                m = mn;
                Z = fmaf(Z, corr, p);
#pragma unroll
                for (int i = 0; i < N; i++) acc[i] = fmaf(p, v.x[i], acc[i] * corr);
            }
            if (__any(is_nan(Z)) || (!stat && point_all(point_nan(acc, nc, j)))) return;
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
template <typename T, int N, int A, bool SEEN> __device__ inline void point_dq(const Args &a, int b, int h, int bh, int ho, int wo, int c0, int nc, bool stat, int lane)
{
    const int j = lane & 15, g = lane >> 4;
    const size_t pq = (size_t)query_point(a, b, ho, ho / a.qps) + (size_t)wo * a.qps, si = ((size_t)bh * a.Ho + ho) * a.Wo + wo;
    PointRow<T, A> q, dy, k, v;
    PointRow<T, N> kc;
    q.load(static_cast<const T *>(a.q) + pq * a.ldq + h * a.dk_, a.dk_, j);
    dy.load(static_cast<const T *>(a.dy) + pq * a.ldg + h * a.dv_, a.dv_, j);
    v.load(static_cast<const T *>(a.ysaved) + pq * a.ldy + h * a.dv_, a.dv_, j);
    const float I = dy.dot(v), lse = a.lse[si];
    bool far = q.far() || dy.far() || v.far() || unusual(lse);
    if (is_nan(I) || is_nan(lse) || is_nan(q.dot(q))) return;
    constexpr bool EXACT_I = std::is_same<T, float>::value;
    float acc[N] = {}, ak[EXACT_I ? 1 : N] = {}, off = 0.f;
    for (int ri = a.goff[ho]; ri < a.goff[ho + 1]; ri++) {
        const Run run = a.gruns[ri];
        const float w = a.quad_w[run.pad];
        const size_t row = (size_t)key_point(a, b, run.lat, run.pad);
        for (int t0 = 0; t0 < run.len; t0 += 4) {
            const bool in = t0 + g < run.len;
            const size_t pk = row + (size_t)((run.ws + wo + t0 + (in ? g : 0)) % a.Wi) * a.kps;
            k.load(static_cast<const T *>(a.k) + pk * a.ldk + h * a.dk_, a.dk_, j);
            v.load(static_cast<const T *>(a.v) + pk * a.ldv + h * a.dv_, a.dv_, j);
            kc.load(static_cast<const T *>(a.k) + pk * a.ldk + h * a.dk_ + c0, nc, j);
            const float p = fast_exp2(fmaf(q.dot(k), LOG2E, -lse)) * w, ds = p * (dy.dot(v) - I);
            if (__any(in && is_nan(ds))) return;
            if (in) {
                far |= k.far() || v.far() || unusual_weight(w);
                if (!EXACT_I) off += ds;
#pragma unroll
                for (int i = 0; i < N; i++) {
                    acc[i] = fmaf(ds, kc.x[i], acc[i]);
                    if (!EXACT_I) ak[EXACT_I ? 0 : i] = fmaf(p, kc.x[i], ak[EXACT_I ? 0 : i]);
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
template <typename T, int N, int A, bool SEEN> __device__ inline void point_dkdv(const Args &a, int b, int h, int bh, int hi, int wi, int c0, int nk, int nv, int lane)
{
    const int j = lane & 15, g = lane >> 4;
    const size_t pk = (size_t)key_point(a, b, hi, hi / a.kps) + (size_t)wi * a.kps;
    PointRow<T, A> k, v, q, dy;
    PointRow<T, N> qc, dyc;
    k.load(static_cast<const T *>(a.k) + pk * a.ldk + h * a.dk_, a.dk_, j);
    v.load(static_cast<const T *>(a.v) + pk * a.ldv + h * a.dv_, a.dv_, j);
    const float w = a.quad_w[hi / a.kps];
    float dk[N] = {}, dv[N] = {};
    bool far = unusual_weight(w) || k.far() || v.far();
    if (is_nan(k.dot(k))) return;
    for (int ri = a.soff[hi]; ri < a.soff[hi + 1]; ri++) {
        const Run run = a.sruns[ri]; // the key is neighbor t of query column wi - ws - t
        const size_t row = (size_t)query_point(a, b, run.lat, run.pad), srow = ((size_t)bh * a.Ho + run.lat) * a.Wo;
        for (int t0 = 0; t0 < run.len; t0 += 4) {
            const bool in = t0 + g < run.len;
            int col = (wi - run.ws - t0 - (in ? g : 0)) % a.Wo;
            col += col < 0 ? a.Wo : 0;
            const size_t pq = row + (size_t)col * a.qps;
            const float2 st = a.stats[srow + col];
            q.load(static_cast<const T *>(a.q) + pq * a.ldq + h * a.dk_, a.dk_, j);
            dy.load(static_cast<const T *>(a.dy) + pq * a.ldg + h * a.dv_, a.dv_, j);
            qc.load(static_cast<const T *>(a.q) + pq * a.ldq + h * a.dk_ + c0, nk, j);
            dyc.load(static_cast<const T *>(a.dy) + pq * a.ldg + h * a.dv_ + c0, nv, j);
            const float p = fast_exp2(fmaf(q.dot(k), LOG2E, -st.x)) * w, ds = p * (dy.dot(v) - st.y);
            if (in) {
                far |= unusual(st.x) || unusual(st.y) || q.far() || dy.far();
#pragma unroll
                for (int i = 0; i < N; i++) {
                    dv[i] = fmaf(p, dyc.x[i], dv[i]);
                    dk[i] = fmaf(ds, qc.x[i], dk[i]);
                }
            }
            if (point_all(point_nan(dv, nv, j) && point_nan(dk, nk, j))) return;
        }
    }
    if (SEEN && !__any(far)) return;
    point_store(static_cast<T *>(a.dk) + pk * a.lddk + h * a.dk_ + c0, dk, 1.f, nk, j, g);
    point_store(static_cast<T *>(a.dv) + pk * a.lddv + h * a.dv_ + c0, dv, 1.f, nv, j, g);
}
