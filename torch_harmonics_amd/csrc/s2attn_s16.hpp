// Matrix-core kernels with the accuracy of fp32 on bf16 matrix instructions: forward, dq and dk/dv, v_mfma_f32_16x16x32_bf16, for fp32
// storage and for the 16-bit head widths that the kernels of s2attn_h16.hpp do not take.
// Included by s2attn_kernels.hip inside namespace s2 after s2attn_h16.hpp, whose tiling they share (a workgroup of four
// wavefronts owns 64 consecutive longitudes of one latitude, 16 per wavefront, and walks its runs in steps of 32 band positions on one
// staged band; lane l = (c = l % 16, qd = l / 16); scores are produced transposed).
//
// fp32 values are split into three bf16 terms when a band row is committed to LDS (split3 in s2attn_split.hpp: |x - h - m - l| <=
// 2^-25 |x|), operands in registers once per workgroup, probabilities once per step; a product is the six term products of at most
// second order.  The five low-order ones go to an accumulator of their own (2^-8 of the other), so the main sum is rounded once per 32
// products: scores, outputs and gradients are closer to float64 than with fp32 matrix instructions.  Six products of 16 clocks for
// 16 x 16 x 32 against eight fp32 instructions of 32 clocks: 2.7 times less matrix time, for 11 vector instructions per two
// staged values, which four wavefronts share.
//
// 16-bit storage: an fp16 value is two bf16 terms, a bf16 value one, both exactly (S terms below); scaled operands, probabilities
// and dS keep three, so nothing between the tensors is rounded to 16 bits, as in the vector kernels.  181 x 360, four heads of
// 20 channels, disk of three spacings, bf16: 86 + 117 + 118 us, 925 + 1128 + 1028 with the vector kernels.
//
// Measured against fp32 matrix instructions (16 longitudes per wavefront, a band each), all three passes: 360 x 720, one head of 64,
// radius 0.03: 1198 -> 970 us; 361 x 720, 16 heads of 64 in all: 16.3 -> 13.9 ms; 181 x 360, eight heads of 48, radius 0.05: 1494 -> 1173
// us (in a tile of 64 channels nothing was gained there).  Against the vector kernels: q, k of 20 and v of 12 channels, 145 x 288:
// 2057 -> 325 us.  The 64-channel kernels are bound by the matrix and vector instructions of the two wavefronts a SIMD holds.
//
// Shape domain: ck and cv multiples of 4, both at most D (zeros are staged past a head's channels and never stored), at least 32
// columns per virtual latitude.  Any point strides; rows need the alignment of four 16-bit values, or of a float.
//
// LDS row of a band: [term][D] bf16; the pitches are 32 or 96 modulo 128 bytes, at which the 16-byte row reads, the
// transposing 8-byte reads and the 16-byte writes are free of bank conflicts.  The band is a ring of FRESH = 80 rows (five blocks of
// 16), all in use in a step: a larger ring would save a barrier per step and cost resident workgroups (64 channels: two per CU).

typedef float f4a __attribute__((ext_vector_type(4), aligned(4)));
typedef unsigned u4a8 __attribute__((ext_vector_type(4), aligned(8)));
typedef unsigned u2a8 __attribute__((ext_vector_type(2), aligned(8)));

// One 16 x 16 block of a sum of split products: hi = sum of h h, lo = the five products of first and second order
struct S16Sum {
    f4v hi, lo;
};
// NX, NY: terms of the operands (those past them are not read)
template <int NX, int NY> __device__ inline void s16_mma(S16Sum &s, const uint4 (&x)[3], const uint4 (&y)[3])
{
    typedef H16<bf16_t> M;
    if (NX > 2) s.lo = M::mfma(x[2], y[0], s.lo);
    s.hi = M::mfma(x[0], y[0], s.hi);
    if (NY > 2) s.lo = M::mfma(x[0], y[2], s.lo);
    if (NX > 1 && NY > 1) s.lo = M::mfma(x[1], y[1], s.lo);
    if (NX > 1) s.lo = M::mfma(x[1], y[0], s.lo);
    if (NY > 1) s.lo = M::mfma(x[0], y[1], s.lo);
}
__device__ inline uint4 s16_u4(u4v x) { return make_uint4(x[0], x[1], x[2], x[3]); }

// eight consecutive values as three packed terms
__device__ inline void s16_split8(uint4 (&o)[3], const float (&x)[8])
{
    u4v t[3];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        unsigned a, b, d;
        split3(x[2 * i], x[2 * i + 1], a, b, d);
        t[0][i] = a, t[1][i] = b, t[2][i] = d;
    }
#pragma unroll
    for (int n = 0; n < 3; n++) o[n] = s16_u4(t[n]);
}
__device__ inline void s16_split_blocks(uint4 (&o)[3], const f4v (&x)[2])
{
    const float f[8] = {x[0][0], x[0][1], x[0][2], x[0][3], x[1][0], x[1][1], x[1][2], x[1][3]};
    s16_split8(o, f);
}

// Eight channels of a grid point in storage type T: S terms are exact.  load: channels `first` .. + 8 of n, zeros past the end.
template <typename T> struct S16Piece {
    static constexpr int S = std::is_same<T, f16_t>::value ? 2 : 1;
    u4v r;
    __device__ inline void zero() { r = u4v{0u, 0u, 0u, 0u}; }
    template <bool PAD> __device__ inline void load(const T *p, int first, int n)
    {
        if (!PAD || first + 8 <= n) {
            r = *reinterpret_cast<const u4a8 *>(p + first);
        } else {
            u2a8 x = {0u, 0u};
            if (first + 4 <= n) x = *reinterpret_cast<const u2a8 *>(p + first);
            r = u4v{x[0], x[1], 0u, 0u};
        }
    }
    __device__ inline void widen(float (&x)[8]) const
    {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float2 f = H16<T>::unpack2(r[i]);
            x[2 * i] = f.x, x[2 * i + 1] = f.y;
        }
    }
};
template <> struct S16Piece<float> {
    static constexpr int S = 3;
    f4a a, b;
    __device__ inline void zero() { a = b = f4a{0.f, 0.f, 0.f, 0.f}; }
    template <bool PAD> __device__ inline void load(const float *p, int first, int n)
    {
        a = b = f4a{0.f, 0.f, 0.f, 0.f};
        if (!PAD || first + 4 <= n) a = *reinterpret_cast<const f4a *>(p + first);
        if (!PAD || first + 8 <= n) b = *reinterpret_cast<const f4a *>(p + first + 4);
    }
    __device__ inline void widen(float (&x)[8]) const
    {
#pragma unroll
        for (int i = 0; i < 4; i++) x[i] = a[i], x[4 + i] = b[i];
    }
};
// S exact terms of a piece (those past S are not written)
template <typename T> __device__ inline void s16_terms(uint4 (&o)[3], const S16Piece<T> &p)
{
    if constexpr (std::is_same<T, bf16_t>::value) {
        o[0] = s16_u4(p.r);
    } else {
        float x[8];
        p.widen(x);
        s16_split8(o, x);
    }
}

__device__ inline void s16_store4(float *p, f4v x) { *reinterpret_cast<f4a *>(p) = x; }
template <typename T> __device__ inline void s16_store4(T *p, f4v x) { *reinterpret_cast<u2a8 *>(p) = u2a8{H16<T>::pack2(x[0], x[1]), H16<T>::pack2(x[2], x[3])}; }

// The band of two tensors: rows of D / 8 pieces of eight channels, one piece per thread, tensor and iteration (48 channels: the last
// four threads take the first pieces of the row after their iteration's, which another thread loads and writes too).
template <int D, int S> constexpr int s16_pitch() { return 2 * S * D + (S * D % 32 ? 0 : 32); }

template <typename T, int D, bool PAD> struct SplitBand {
    static constexpr int S = S16Piece<T>::S, PITCH = s16_pitch<D, S>();
    static constexpr int CPR = D / 8, RPI = 64 * NW / CPR, NIT = (FRESH + RPI - 1) / RPI;
    static constexpr int BYTES = FRESH * PITCH;
    S16Piece<T> ra[NIT], rb[NIT];

    // rows cs .. cs + N (columns of the circle, 0 <= cs < W) of pa, pb; columns lda, ldb elements apart; na, nb channels
    template <int N> __device__ inline void fetch(const T *pa, const T *pb, int tid, int cs, int W, unsigned lda, unsigned ldb, int na, int nb)
    {
        const int r0 = tid / CPR, ch = 8 * (tid % CPR);
#pragma unroll
        for (int it = 0; it < (N + RPI - 1) / RPI; it++) {
            if ((it + 1) * RPI <= N || it * RPI + r0 < N) {
                unsigned col = (unsigned)(cs + it * RPI + r0);
                col = min(col, col - (unsigned)W); // (wraps to a huge value when col < W)
                if (W < FRESH) col = min(col, col - (unsigned)W), col = min(col, col - (unsigned)W);
                ra[it].template load<PAD>(pa + col * lda, ch, na);
                rb[it].template load<PAD>(pb + col * ldb, ch, nb);
            }
        }
    }
    // The same for rows lo .. hi of N, zeros elsewhere (a ring step's band is clipped): row lo is column `col` of pa, pb, columns ld elements
    // apart; wrap > 0: the number of columns the later rows wrap around (at least 32; col + hi - lo < 4 wrap)
    template <int N> __device__ inline void fetch_rows(const T *pa, const T *pb, int tid, int lo, int hi, unsigned ld, int n, int col = 0, int wrap = 0)
    {
        const int r0 = tid / CPR, ch = 8 * (tid % CPR);
#pragma unroll
        for (int it = 0; it < (N + RPI - 1) / RPI; it++) {
            if ((it + 1) * RPI <= N || it * RPI + r0 < N) {
                const int r = it * RPI + r0;
                ra[it].zero();
                rb[it].zero();
                if (r >= lo && r < hi) {
                    unsigned x = (unsigned)(col + r - lo);
                    if (wrap) x = min(x, x - (unsigned)wrap), x = min(x, x - (unsigned)wrap), x = min(x, x - (unsigned)wrap);
                    ra[it].template load<PAD>(pa + (size_t)x * ld, ch, n);
                    rb[it].template load<PAD>(pb + (size_t)x * ld, ch, n);
                }
            }
        }
    }
    // the N rows fetched last become ring rows x0 .. x0 + N (modulo the ring), those of the first tensor times log2 e if SCALED (fp32)
    template <int N, bool SCALED = false> __device__ inline void commit(char *A, char *B, int tid, int x0)
    {
        const int r0 = tid / CPR, pc = 16 * (tid % CPR);
#pragma unroll
        for (int it = 0; it < (N + RPI - 1) / RPI; it++) {
            if ((it + 1) * RPI <= N || it * RPI + r0 < N) {
                int r = x0 + it * RPI + r0;
                r -= r >= FRESH ? FRESH : 0;
                if constexpr (SCALED) ra[it].a *= LOG2E, ra[it].b *= LOG2E;
                uint4 t[3];
                s16_terms<T>(t, ra[it]);
#pragma unroll
                for (int n = 0; n < S; n++) *reinterpret_cast<uint4 *>(A + r * PITCH + 2 * D * n + pc) = t[n];
                s16_terms<T>(t, rb[it]);
#pragma unroll
                for (int n = 0; n < S; n++) *reinterpret_cast<uint4 *>(B + r * PITCH + 2 * D * n + pc) = t[n];
            }
        }
    }
};

// The lane's own operand of a score product (a grid point's vector; this lane supplies channels 32 s + 8 qd .. + 8 of instruction s),
// as it is (NT = S terms) or times log2 e (three terms).  Heads of up to 16 channels fill the 32 k slots of an instruction with two terms.
// Three staged terms: rows [h m] against [h h] and [m m], rows [l h] against [h l] are all six products.  Two: rows [h m] against
// [h h], [m m] and [l l].  One: rows [h h] against [h m] and [l 0].
template <typename T, int D, bool SCALED> struct S16Own {
    static constexpr int S = S16Piece<T>::S, NT = SCALED ? 3 : S;
    static constexpr int NS = (D + 31) / 32;
    uint4 t[NS][3];
    template <bool PAD> __device__ inline void load(const T *p, int n, int qd)
    {
#pragma unroll
        for (int s = 0; s < NS; s++) {
            S16Piece<T> r;
            r.template load<PAD>(p, D == 16 ? 8 * (qd & 1) : 32 * s + 8 * qd, n);
            float x[8];
            r.widen(x);
            if (SCALED) {
#pragma unroll
                for (int i = 0; i < 8; i++) x[i] *= LOG2E;
            }
            s16_split8(t[s], x);
        }
        if (D == 16 && S == 3 && qd < 2) t[0][2] = t[0][0];
        if (D == 16 && S == 1) {
            const uint4 zero = make_uint4(0u, 0u, 0u, 0u);
            if (qd >= 2) t[0][0] = t[0][1], t[0][2] = zero;
            t[0][1] = t[0][2];
        }
    }
    __device__ inline void settle_()
    {
#pragma unroll
        for (int s = 0; s < NS; s++) settle(t[s]);
    }
};

// sum += (rows of the 16-row block) x own: the lane's block of scores, rows 4 qd + v, column c
template <typename T, int D, bool SCALED> __device__ inline void s16_scores(S16Sum &sum, const char *blk, int c, int qd, const S16Own<T, D, SCALED> &own)
{
    typedef H16<bf16_t> M;
    constexpr int S = S16Piece<T>::S;
    const char *row = blk + c * s16_pitch<D, S>();
    if constexpr (D == 16) {
        const uint4 hm = *reinterpret_cast<const uint4 *>(row + (S == 1 ? 16 * (qd & 1) : 16 * qd));
        if constexpr (S == 3) {
            const uint4 lh = *reinterpret_cast<const uint4 *>(row + (qd < 2 ? 64 + 16 * qd : 16 * qd - 32));
            sum.lo = M::mfma(lh, own.t[0][2], sum.lo);
        } else if constexpr (S == 2 && SCALED) {
            sum.lo = M::mfma(hm, own.t[0][2], sum.lo);
        }
        sum.hi = M::mfma(hm, own.t[0][0], sum.hi);
        if (S > 1 || SCALED) sum.lo = M::mfma(hm, own.t[0][1], sum.lo);
    } else {
#pragma unroll
        for (int s = 0; s < (D + 31) / 32; s++) {
            uint4 x[3];
            // (48 channels: the upper half of the last instruction has zeros on the other side)
            const char *piece = row + 64 * s + 16 * (32 * s + 32 <= D ? qd : qd & 1);
#pragma unroll
            for (int n = 0; n < S; n++) x[n] = *reinterpret_cast<const uint4 *>(piece + 2 * D * n);
            s16_mma<S, S16Own<T, D, SCALED>::NT>(sum, x, own.t[s]);
        }
    }
}

// acc[cb] (channels 16 cb + 4 qd + v of column c) += sum over the 32 rows of two blocks of row[channel] * coefficient
template <int D, int S> __device__ inline void s16_accumulate(S16Sum (&acc)[D / 16], const char *blk0, const char *blk1, int c, int qd, const uint4 (&p)[3])
{
#pragma unroll
    for (int cb = 0; cb < D / 16; cb++) {
        uint4 x[3];
#pragma unroll
        for (int n = 0; n < S; n++) x[n] = h16_read_transposed<s16_pitch<D, S>()>(blk0 + 2 * D * n, blk1 + 2 * D * n, cb, c, qd);
        s16_mma<S, 3>(acc[cb], x, p);
    }
}

// The same into one sum per block: the low-order products of the 32 rows are added up first and then added to it.  Four more vector
// additions per block and step, half the registers: for the dk/dv pass of 64 channels, which spills otherwise.
template <int D, int S> __device__ inline void s16_accumulate(f4v (&acc)[D / 16], const char *blk0, const char *blk1, int c, int qd, const uint4 (&p)[3])
{
#pragma unroll
    for (int cb = 0; cb < D / 16; cb++) {
        uint4 x[3];
#pragma unroll
        for (int n = 0; n < S; n++) x[n] = h16_read_transposed<s16_pitch<D, S>()>(blk0 + 2 * D * n, blk1 + 2 * D * n, cb, c, qd);
        S16Sum t = {acc[cb], f4v{0.f, 0.f, 0.f, 0.f}};
        s16_mma<S, 3>(t, x, p);
        acc[cb] = t.hi + t.lo;
    }
}

__device__ inline f4v s16_value(const S16Sum &s) { return s.hi + s.lo; }
__device__ inline f4v s16_value(const f4v &s) { return s; }
template <int N> __device__ inline void s16_zero(f4v (&acc)[N])
{
#pragma unroll
    for (int i = 0; i < N; i++) acc[i] = f4v{0.f, 0.f, 0.f, 0.f};
}
template <int N> __device__ inline void s16_zero(S16Sum (&acc)[N])
{
#pragma unroll
    for (int i = 0; i < N; i++) acc[i].hi = acc[i].lo = f4v{0.f, 0.f, 0.f, 0.f};
}

// Start values of a step's two blocks of scores: `start` where the element is a neighbor, -inf (a probability of zero) elsewhere.
// Element (kb, v) of a lane is neighbor tb + pos + 16 kb + v of its column, tb = 4 qd - c; only the first step of a run
// has elements before the first neighbor.
__device__ inline void s16_start(S16Sum (&sc)[2], int tb, int pos, int len, float start)
{
    sc[0].lo = sc[1].lo = f4v{0.f, 0.f, 0.f, 0.f};
    if (pos >= HQ - 1 && pos + HK <= len) {
        sc[0].hi = sc[1].hi = f4v{start, start, start, start};
    } else if (pos == 0) {
#pragma unroll
        for (int kb = 0; kb < 2; kb++)
#pragma unroll
            for (int v = 0; v < 4; v++) sc[kb].hi[v] = (unsigned)(tb + 16 * kb + v) < (unsigned)len ? start : -INFINITY;
    } else {
#pragma unroll
        for (int kb = 0; kb < 2; kb++)
#pragma unroll
            for (int v = 0; v < 4; v++) sc[kb].hi[v] = tb + 16 * kb + v < len - pos ? start : -INFINITY;
    }
}

template <typename T, int D> constexpr int s16_lds_bytes(bool stats) { return 2 * SplitBand<T, D, false>::BYTES + (stats ? FRESH * 8 : 0); }

// block of the ring `n` blocks after block `first` (both below 5)
__device__ inline int s16_block(int first, int n) { return first + n >= FRESH / 16 ? first + n - FRESH / 16 : first + n; }

// The columns `redo` of a wavefront whose sums are not finite, stored already (see s2attn_points.hpp)
template <typename T, int D, bool PAD, Which PASS> __device__ __forceinline__ void s16_points(int wv, unsigned redo)
{
    constexpr int N = D / 16;
    constexpr bool SEEN = std::is_same<T, float>::value && D == 32 && !PAD;
    __threadfence(); // what is written here comes after it
    const Args a = point_args();
    S2_H16_IDS_OF(64 * wv + point_lane(), blockIdx.x, PASS == DKDV ? a.Wi : a.Wo, PASS == DKDV ? a.Hi : a.Ho)
    (void)c, (void)qd, (void)nvalid;
    const int row = (PASS == DKDV ? a.sorder : a.gorder)[a.row_first + rowsel];
    for (; redo; redo &= redo - 1) {
        const int col = w0 + __builtin_ctz(redo);
        if (PASS == FWD) point_forward<T, N, N, SEEN>(a, b, h, bh, row, col, 0, a.dv_, true, lane);
        if (PASS == DQ) point_dq<T, N, N, SEEN>(a, b, h, bh, row, col, 0, a.dk_, true, lane);
        if (PASS == DKDV) point_dkdv<T, N, N, SEEN>(a, b, h, bh, row, col, 0, a.dk_, a.dv_, lane);
    }
}

// ---- forward ---------------------------------------------------------------------------------------------------
template <typename T, int D, bool PAD> __global__ __launch_bounds__(64 * NW) void fwd_s16_kernel(const Args a)
{
    typedef SplitBand<T, D, PAD> Band_;
    constexpr int S = Band_::S, PITCH = Band_::PITCH, NCB = D / 16;
    extern __shared__ __attribute__((aligned(16))) char h16_lds[];
    char *Ks = h16_lds, *Vs = h16_lds + Band_::BYTES;

    S2_H16_IDS(a.Wo, a.Ho)
    const int wv = __builtin_amdgcn_readfirstlane(wave);
    const int ho = a.gorder[a.row_first + rowsel];
    const int nk = PAD ? a.dk_ : D, nv = PAD ? a.dv_ : D;
    const T *kx = static_cast<const T *>(a.k) + (size_t)b * a.Hi * a.Wi * a.ldk + h * nk;
    const T *vx = static_cast<const T *>(a.v) + (size_t)b * a.Hi * a.Wi * a.ldv + h * nv;
    const bool mine = c < nvalid;
    const size_t pt = (size_t)query_point(a, b, ho, ho / a.qps) + (size_t)(w0 + (mine ? c : 0)) * a.qps;

    S16Own<T, D, true> own; // q log2 e: scores come out in the log2 domain
    own.template load<PAD>(static_cast<const T *>(a.q) + pt * a.ldq + h * nk, nk, qd);
    S16Sum acc[NCB]; // Y^T: register v of block cb is channel 16 cb + 4 qd + v of column c
    s16_zero(acc);
    float m = 0.f, Z = 0.f;
    bool first = true; // this column has seen no neighbor of positive weight

    H16Walk wk;
    wk.ri = a.goff[ho];
    wk.rend = a.goff[ho + 1];
    wk.pos = 0;
    wk.run = Run{0, 0, 0, 0};
    Band_ bd;
    const unsigned lda = a.ldk * a.kps, ldb = a.ldv * a.kps; // elements between two columns of a virtual input latitude
    auto fetch = [&](const Run &rn, bool fresh) {
        const size_t row = (size_t)key_row(a, rn.lat, rn.pad);
        const int cs = wk.stage(fresh, rn.ws + wg0, a.Wi);
        if (fresh)
            bd.template fetch<FRESH>(kx + row * a.ldk, vx + row * a.ldv, tid, cs, a.Wi, lda, ldb, nk, nv);
        else
            bd.template fetch<HK>(kx + row * a.ldk, vx + row * a.ldv, tid, cs, a.Wi, lda, ldb, nk, nv);
    };
    wk.w = 1.f;
    if (wk.ri < wk.rend) {
        wk.run = a.gruns[wk.ri];
        wk.w = a.quad_w[wk.run.pad];
        fetch(wk.run, true);
        bd.template commit<FRESH>(Ks, Vs, tid, 0);
    }
    __syncthreads();
    own.settle_();

    const int tb = 4 * qd - c;
    int rb = 0; // ring block of band position `pos`
    while (wk.ri < wk.rend) {
        wk.plan(a.gruns, a.quad_w);
        if (wk.more) fetch(wk.nrun, wk.fresh);
        if (active) {
            const int b0 = s16_block(rb, wv), b1 = s16_block(b0, 1);
            const char *k0 = Ks + b0 * 16 * PITCH, *k1 = Ks + b1 * 16 * PITCH, *v0 = Vs + b0 * 16 * PITCH, *v1 = Vs + b1 * 16 * PITCH;
            // The sums start at log2 w - m, so they end as the exponents of the probabilities.
            S16Sum sc[2];
            s16_start(sc, tb, wk.pos, wk.run.len, fast_log2(wk.w) - m);
            s16_scores(sc[0], k0, c, qd, own);
            s16_scores(sc[1], k1, c, qd, own);
            f4v p[2] = {sc[0].hi + sc[0].lo, sc[1].hi + sc[1].lo};
            float mx = fmaxf(fmaxf(fmaxf(p[0][0], p[0][1]), fmaxf(p[0][2], p[0][3])), fmaxf(fmaxf(p[1][0], p[1][1]), fmaxf(p[1][2], p[1][3])));
            // The running maximum is only the reference point of the exponentials: it moves when a column's maximum has
            // grown by more than RESCALE_THR (probabilities stay below 2^RESCALE_THR), which after a row's first steps is rare.
            // A column's first step with a neighbor always sets it.  (Every column has a neighbor in the first step of a run, but on a
            // latitude of quadrature weight 0 its maximum is -inf, which is no reference point.)
            if (__any(first || mx > RESCALE_THR)) {
                const float cm = h16_quarter_max(mx);
                const float d = (first && cm > -INFINITY) || cm > RESCALE_THR ? cm : 0.f;
                const float corr = first ? 0.f : fast_exp2(-d);
                Z *= corr;
#pragma unroll
                for (int cb = 0; cb < NCB; cb++) acc[cb].hi *= corr, acc[cb].lo *= corr;
                p[0] -= d, p[1] -= d;
                m += d;
                first = first && !(cm > -INFINITY);
            }
#pragma unroll
            for (int kb = 0; kb < 2; kb++) {
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    p[kb][v] = fast_exp2(p[kb][v]); // masked: exp2(-inf) = 0
                    Z += p[kb][v];                  // this lane's share; the four lanes of a column are added up at the end
                }
            }
            uint4 ps[3];
            s16_split_blocks(ps, p);
            s16_accumulate<D, S>(acc, v0, v1, c, qd, ps);
        }
        if (wk.more) {
            __syncthreads(); // the next rows replace rows the slowest wavefront may still be reading
            rb = wk.fresh ? 0 : s16_block(rb, 2);
            if (wk.fresh)
                bd.template commit<FRESH>(Ks, Vs, tid, 0);
            else
                bd.template commit<HK>(Ks, Vs, tid, 16 * s16_block(rb, 3));
        }
        __syncthreads();
        wk.advance();
    }

    Z = h16_quarter_sum(Z);
    float check = Z;
#pragma unroll
    for (int cb = 0; cb < NCB; cb++) check += point_sum(acc[cb].hi + acc[cb].lo);
    const unsigned redo = point_columns(mine && not_finite(check));
    if (mine) {
        if (a.lse && qd == 0) a.lse[((size_t)bh * a.Ho + ho) * a.Wo + w0 + c] = m + fast_log2(Z);
        const float inv = 1.0f / Z;
        T *y = static_cast<T *>(a.y) + pt * a.ldy + h * nv + 4 * qd;
#pragma unroll
        for (int cb = 0; cb < NCB; cb++)
            if (!PAD || 16 * cb + 4 * qd < nv) s16_store4(y + 16 * cb, (acc[cb].hi + acc[cb].lo) * inv);
    }
    if (__builtin_expect(redo != 0, 0)) s16_points<T, D, PAD, FWD>(wv, redo);
}

// ---- backward, dq pass (needs the forward's y and lse) -------------------------------------------------------------
// Three products per step:  S^T = K Q^T,  G^T = V dY^T,  dQ^T += K^T dS^T  with dS = P o (G - I),  I = <dy, y>.
// 16-bit storage: the stored y is rounded, so I is only a first value of the mean of G.  The walk adds up how far the mean is from it,
// sum P (G - I) (at most 2^-9 of it), and AK = sum P k from the leading term of P, and dq takes the product of the two off at the end.
template <typename T, int D, bool PAD> __global__ __launch_bounds__(64 * NW) void dq_s16_kernel(const Args a)
{
    typedef SplitBand<T, D, PAD> Band_;
    constexpr int S = Band_::S, PITCH = Band_::PITCH, NCB = D / 16;
    extern __shared__ __attribute__((aligned(16))) char h16_lds[];
    char *Ks = h16_lds, *Vs = h16_lds + Band_::BYTES;

    S2_H16_IDS(a.Wo, a.Ho)
    const int wv = __builtin_amdgcn_readfirstlane(wave);
    const int ho = a.gorder[a.row_first + rowsel];
    const int nk = PAD ? a.dk_ : D, nv = PAD ? a.dv_ : D;
    const T *kx = static_cast<const T *>(a.k) + (size_t)b * a.Hi * a.Wi * a.ldk + h * nk;
    const T *vx = static_cast<const T *>(a.v) + (size_t)b * a.Hi * a.Wi * a.ldv + h * nv;
    const bool mine = c < nvalid;
    const size_t pt = (size_t)query_point(a, b, ho, ho / a.qps) + (size_t)(w0 + (mine ? c : 0)) * a.qps;
    const size_t sidx = ((size_t)bh * a.Ho + ho) * a.Wo + w0 + (mine ? c : 0);

    S16Own<T, D, true> qo;
    S16Own<T, D, false> go;
    qo.template load<PAD>(static_cast<const T *>(a.q) + pt * a.ldq + h * nk, nk, qd);
    const T *dyp = static_cast<const T *>(a.dy) + pt * a.ldg + h * nv;
    go.template load<PAD>(dyp, nv, qd);
    float I = 0.f;
    {
        const T *yp = static_cast<const T *>(a.ysaved) + pt * a.ldy + h * nv;
#pragma unroll
        for (int s = 0; s < (D + 31) / 32; s++) {
            S16Piece<T> yr, gr;
            yr.template load<PAD || D == 16>(yp, 32 * s + 8 * qd, nv); // (16 channels: the upper two quarters have none)
            gr.template load<PAD || D == 16>(dyp, 32 * s + 8 * qd, nv);
            float x[8], g[8];
            yr.widen(x);
            gr.widen(g);
#pragma unroll
            for (int i = 0; i < 8; i++) I = fmaf(g[i], x[i], I);
        }
    }
    I = h16_quarter_sum(I);
    const float lse = a.lse[sidx];

    S16Sum acc[NCB];
    s16_zero(acc);
    constexpr bool EXACT_I = S == 3;
    f4v ak[EXACT_I ? 1 : NCB];
    s16_zero(ak);
    float off = 0.f;

    H16Walk wk;
    wk.ri = a.goff[ho];
    wk.rend = a.goff[ho + 1];
    wk.pos = 0;
    wk.run = Run{0, 0, 0, 0};
    Band_ bd;
    const unsigned lda = a.ldk * a.kps, ldb = a.ldv * a.kps;
    auto fetch = [&](const Run &rn, bool fresh) {
        const size_t row = (size_t)key_row(a, rn.lat, rn.pad);
        const int cs = wk.stage(fresh, rn.ws + wg0, a.Wi);
        if (fresh)
            bd.template fetch<FRESH>(kx + row * a.ldk, vx + row * a.ldv, tid, cs, a.Wi, lda, ldb, nk, nv);
        else
            bd.template fetch<HK>(kx + row * a.ldk, vx + row * a.ldv, tid, cs, a.Wi, lda, ldb, nk, nv);
    };
    wk.w = 1.f;
    if (wk.ri < wk.rend) {
        wk.run = a.gruns[wk.ri];
        wk.w = a.quad_w[wk.run.pad];
        fetch(wk.run, true);
        bd.template commit<FRESH>(Ks, Vs, tid, 0);
    }
    __syncthreads();
    qo.settle_();
    go.settle_();
    float lse_ = lse;
    settle(lse_);

    const int tb = 4 * qd - c;
    int rb = 0;
    while (wk.ri < wk.rend) {
        wk.plan(a.gruns, a.quad_w);
        if (wk.more) fetch(wk.nrun, wk.fresh);
        if (active) {
            const int b0 = s16_block(rb, wv), b1 = s16_block(b0, 1);
            const char *k0 = Ks + b0 * 16 * PITCH, *k1 = Ks + b1 * 16 * PITCH, *v0 = Vs + b0 * 16 * PITCH, *v1 = Vs + b1 * 16 * PITCH;
            // The sums start at log2 w - lse and at -I, so they end as the exponent of p and as g - I.
            S16Sum sc[2], gc[2];
            s16_start(sc, tb, wk.pos, wk.run.len, fast_log2(wk.w) - lse_);
            gc[0].hi = gc[1].hi = f4v{-I, -I, -I, -I};
            gc[0].lo = gc[1].lo = f4v{0.f, 0.f, 0.f, 0.f};
            s16_scores(sc[0], k0, c, qd, qo);
            s16_scores(sc[1], k1, c, qd, qo);
            s16_scores(gc[0], v0, c, qd, go);
            s16_scores(gc[1], v1, c, qd, go);
            f4v p[2], ds[2];
#pragma unroll
            for (int kb = 0; kb < 2; kb++)
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    p[kb][v] = fast_exp2(sc[kb].hi[v] + sc[kb].lo[v]);
                    ds[kb][v] = p[kb][v] * (gc[kb].hi[v] + gc[kb].lo[v]);
                    if (!EXACT_I) off += ds[kb][v];
                }
            if constexpr (!EXACT_I) {
                const uint4 pb = make_uint4(pk_bf16(p[0][0], p[0][1]), pk_bf16(p[0][2], p[0][3]), pk_bf16(p[1][0], p[1][1]), pk_bf16(p[1][2], p[1][3]));
#pragma unroll
                for (int cb = 0; cb < NCB; cb++) ak[cb] = H16<bf16_t>::mfma(h16_read_transposed<PITCH>(k0, k1, cb, c, qd), pb, ak[cb]);
            }
            uint4 ps[3];
            s16_split_blocks(ps, ds);
            s16_accumulate<D, S>(acc, k0, k1, c, qd, ps);
        }
        if (wk.more) {
            __syncthreads();
            rb = wk.fresh ? 0 : s16_block(rb, 2);
            if (wk.fresh)
                bd.template commit<FRESH>(Ks, Vs, tid, 0);
            else
                bd.template commit<HK>(Ks, Vs, tid, 16 * s16_block(rb, 3));
        }
        __syncthreads();
        wk.advance();
    }

    // (stored after the walk: a global store ahead of the loop would turn the loop's scalar loads of runs and weights,
    // which the compiler only uses while nothing in the kernel can have written memory, into vector loads with waits)
    off = EXACT_I ? 0.f : h16_quarter_sum(off);
    float check = off;
#pragma unroll
    for (int cb = 0; cb < NCB; cb++) check += point_sum(EXACT_I ? acc[cb].hi + acc[cb].lo : acc[cb].hi + acc[cb].lo + ak[EXACT_I ? 0 : cb]);
    const unsigned redo = point_columns(mine && not_finite(check));
    if (mine) {
        if (qd == 0) a.stats[sidx] = make_float2(lse, I + off);
        T *dq = static_cast<T *>(a.dq) + pt * a.lddq + h * nk + 4 * qd;
#pragma unroll
        for (int cb = 0; cb < NCB; cb++)
            if (!PAD || 16 * cb + 4 * qd < nk) s16_store4(dq + 16 * cb, EXACT_I ? acc[cb].hi + acc[cb].lo : (acc[cb].hi + acc[cb].lo) - off * ak[EXACT_I ? 0 : cb]);
    }
    if (__builtin_expect(redo != 0, 0)) s16_points<T, D, PAD, DQ>(wv, redo);
}

// ---- backward, dk/dv pass: transposed gather ---------------------------------------------------------------------
// The wavefront owns 16 INPUT longitudes (column c = key) and walks the runs grouped by input latitude; staged rows
// are queries.  Staged row r of a run (first row = longitude w0 - ws - len + 1) sees key c iff 0 <= r - c < len.
// Four products per step:  S = Q K^T,  G = dY V^T  (rows = queries, columns = keys),  dV^T += dY^T P,  dK^T += Q^T dS.
// fp32: q is staged times log2 e, rounded as the other two passes round it, so all three see the same scores (the gradients lean on
// sums of dS that cancel exactly: q (k log2 e) instead doubles the noise in sum dk); dk takes the factor back at the end.  16-bit: q is
// staged as it is, an exact term or two, and k carries the factor.
template <typename T, int D, bool PAD> __global__ __launch_bounds__(64 * NW, D == 64 || (D == 48 && S16Piece<T>::S == 3) ? 2 : (D == 32 && S16Piece<T>::S == 1 ? 4 : 3)) void dkdv_s16_kernel(const Args a)
{
    typedef SplitBand<T, D, PAD> Band_;
    constexpr int S = Band_::S, PITCH = Band_::PITCH, NCB = D / 16;
    extern __shared__ __attribute__((aligned(16))) char h16_lds[];
    char *Qs = h16_lds, *Gs = h16_lds + Band_::BYTES;
    float2 *Ts = reinterpret_cast<float2 *>(h16_lds + 2 * Band_::BYTES); // (log2 w - lse, -I) of the staged queries

    S2_H16_IDS(a.Wi, a.Hi)
    const int wv = __builtin_amdgcn_readfirstlane(wave);
    const int hi = a.sorder[a.row_first + rowsel];
    const int nk = PAD ? a.dk_ : D, nv = PAD ? a.dv_ : D;
    const T *qy = static_cast<const T *>(a.q) + (size_t)b * a.Ho * a.Wo * a.ldq + h * nk;
    const T *gy = static_cast<const T *>(a.dy) + (size_t)b * a.Ho * a.Wo * a.ldg + h * nv;
    const float2 *stats = a.stats + (size_t)bh * a.Ho * a.Wo;
    const bool mine = c < nvalid;
    const size_t pt = (size_t)key_point(a, b, hi, hi / a.kps) + (size_t)(w0 + (mine ? c : 0)) * a.kps;

    constexpr bool QSCALED = S == 3;
    S16Own<T, D, !QSCALED> ko;
    S16Own<T, D, false> vo;
    ko.template load<PAD>(static_cast<const T *>(a.k) + pt * a.ldk + h * nk, nk, qd);
    vo.template load<PAD>(static_cast<const T *>(a.v) + pt * a.ldv + h * nv, nv, qd);
    typename std::conditional<(D >= 32), f4v, S16Sum>::type dkt[NCB], dvt[NCB];
    s16_zero(dkt);
    s16_zero(dvt);
    const float lw = fast_log2(a.quad_w[hi / a.kps]);

    H16Walk wk;
    wk.ri = a.soff[hi];
    wk.rend = a.soff[hi + 1];
    wk.pos = 0;
    wk.run = Run{0, 0, 0, 0};
    wk.w = 1.f;
    Band_ bd;
    float2 st = make_float2(0.f, 0.f);
    const unsigned lda = a.ldq * a.qps, ldb = a.ldg * a.qps; // elements between two columns of a virtual output latitude
    auto fetch = [&](const Run &rn, bool fresh) {
        int c0 = 0;
        if (fresh) { // longitude of band row 0, in [0, 2 W)
            c0 = wg0 - rn.ws - rn.len + 1 + a.Wo;
            while (c0 < 0) c0 += a.Wo;
        }
        const int cs = wk.stage(fresh, c0, a.Wo);
        const size_t row = (size_t)query_row(a, rn.lat, rn.pad);
        if (fresh)
            bd.template fetch<FRESH>(qy + row * a.ldq, gy + row * a.ldg, tid, cs, a.Wo, lda, ldb, nk, nv);
        else
            bd.template fetch<HK>(qy + row * a.ldq, gy + row * a.ldg, tid, cs, a.Wo, lda, ldb, nk, nv);
        if (tid < (fresh ? FRESH : HK)) { // the first threads fetch the statistics of the staged rows
            int col = cs + tid;
            while (col >= a.Wo) col -= a.Wo;
            st = stats[(size_t)rn.lat * a.Wo + col];
        }
    };
    auto commit = [&](bool fresh, int x0) {
        if (fresh)
            bd.template commit<FRESH, QSCALED>(Qs, Gs, tid, 0);
        else
            bd.template commit<HK, QSCALED>(Qs, Gs, tid, x0);
        if (tid < (fresh ? FRESH : HK)) {
            int r = x0 + tid;
            r -= r >= FRESH ? FRESH : 0;
            Ts[r] = make_float2(lw - st.x, -st.y);
        }
    };
    if (wk.ri < wk.rend) {
        wk.run = a.sruns[wk.ri];
        fetch(wk.run, true);
        commit(true, 0);
    }
    __syncthreads();
    ko.settle_();
    vo.settle_();

    const int tb = 4 * qd - c;
    int rb = 0;
    while (wk.ri < wk.rend) {
        wk.plan(a.sruns);
        if (wk.more) fetch(wk.nrun, wk.fresh);
        if (active) {
            const int len = wk.run.len, pos = wk.pos;
            const int blk[2] = {s16_block(rb, wv), s16_block(s16_block(rb, wv), 1)};
            const char *q0 = Qs + blk[0] * 16 * PITCH, *q1 = Qs + blk[1] * 16 * PITCH, *g0 = Gs + blk[0] * 16 * PITCH, *g1 = Gs + blk[1] * 16 * PITCH;
            // The sums start at the staged statistics, so they end as the exponent of p and as g - I.
            S16Sum sc[2], gc[2];
#pragma unroll
            for (int qb = 0; qb < 2; qb++) {
                const float4 *sp = reinterpret_cast<const float4 *>(Ts + 16 * blk[qb] + 4 * qd);
                const float4 s01 = sp[0], s23 = sp[1];
                sc[qb].hi = f4v{s01.x, s01.z, s23.x, s23.z};
                gc[qb].hi = f4v{s01.y, s01.w, s23.y, s23.w};
                sc[qb].lo = gc[qb].lo = f4v{0.f, 0.f, 0.f, 0.f};
            }
            if (pos == 0) { // (rows outside the neighborhood: a probability of zero)
#pragma unroll
                for (int qb = 0; qb < 2; qb++)
#pragma unroll
                    for (int v = 0; v < 4; v++) sc[qb].hi[v] = (unsigned)(tb + 16 * qb + v) < (unsigned)len ? sc[qb].hi[v] : -INFINITY;
            } else if (pos + HK > len) {
#pragma unroll
                for (int qb = 0; qb < 2; qb++)
#pragma unroll
                    for (int v = 0; v < 4; v++) sc[qb].hi[v] = tb + 16 * qb + v < len - pos ? sc[qb].hi[v] : -INFINITY;
            }
            s16_scores(sc[0], q0, c, qd, ko);
            s16_scores(sc[1], q1, c, qd, ko);
            s16_scores(gc[0], g0, c, qd, vo);
            s16_scores(gc[1], g1, c, qd, vo);
            f4v p[2], ds[2];
#pragma unroll
            for (int qb = 0; qb < 2; qb++)
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    p[qb][v] = fast_exp2(sc[qb].hi[v] + sc[qb].lo[v]);
                    ds[qb][v] = p[qb][v] * (gc[qb].hi[v] + gc[qb].lo[v]);
                }
            uint4 ps[3];
            s16_split_blocks(ps, p);
            s16_accumulate<D, S>(dvt, g0, g1, c, qd, ps);
            s16_split_blocks(ps, ds);
            s16_accumulate<D, S>(dkt, q0, q1, c, qd, ps);
        }
        if (wk.more) {
            __syncthreads();
            rb = wk.fresh ? 0 : s16_block(rb, 2);
            commit(wk.fresh, wk.fresh ? 0 : 16 * s16_block(rb, 3));
        }
        __syncthreads();
        wk.advance();
    }

    float check = 0.f;
#pragma unroll
    for (int cb = 0; cb < NCB; cb++) check += point_sum(s16_value(dkt[cb]) + s16_value(dvt[cb]));
    const unsigned redo = point_columns(mine && not_finite(check));
    if (mine) {
        T *dk = static_cast<T *>(a.dk) + pt * a.lddk + h * nk + 4 * qd, *dv = static_cast<T *>(a.dv) + pt * a.lddv + h * nv + 4 * qd;
#pragma unroll
        for (int cb = 0; cb < NCB; cb++) {
            if (!PAD || 16 * cb + 4 * qd < nk) s16_store4(dk + 16 * cb, s16_value(dkt[cb]) * (QSCALED ? 1.f / LOG2E : 1.f));
            if (!PAD || 16 * cb + 4 * qd < nv) s16_store4(dv + 16 * cb, s16_value(dvt[cb]));
        }
    }
    if (__builtin_expect(redo != 0, 0)) s16_points<T, D, PAD, DKDV>(wv, redo);
}
