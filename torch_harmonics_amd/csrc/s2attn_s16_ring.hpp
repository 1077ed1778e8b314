// Ring steps of a longitude-sharded layer on split products: forward, pass 1 and pass 2 for heads of 17 to 64 channels
// (which storage and sizes: ring_split in s2attn_kernels.hip, with both sides' times).
// Included by s2attn_kernels.hip inside namespace s2 after s2attn_s16.hpp (tiles, split products, band in LDS) and s2attn_m32.hpp
// (the ring steps for the other heads, whose state, modes and clipping these kernels share).
//
// What bounds a ring step: on long runs the matrix and vector work of its tile steps, on short ones a run's chain of loads, barrier and
// one or two steps; the caller's state is read and written once.  All three passes: 721 x 1440, eight heads of 32, four chunks, bf16: 10.9 ms
// with fp32 matrix instructions on widened values, 5.6 here; 361 x 720, two batches of four heads of 64, radius 0.044, two chunks: 16.9 ms,
// 6.1 here.  State and gradients are as close to float64 as there or closer (relative 2-norm of y_acc 2.7e-7 for 3.1e-7, dk 2.1e-7 for 2.3e-7).
//
// A workgroup of four wavefronts owns 64 consecutive longitudes.  Row x of its band of a run is the grid point "workgroup's first
// longitude + run start + x"; the chunk (pass 2: the window of local queries) clips ROWS, so of a run's band up to three intervals
// [ua, ub) of rows are staged, rows beyond them as zeros.  Wavefront w stands at rows 16 w + pos .. + 32, so the walk of an interval
// starts 48 positions early, and a wavefront whose 32 rows miss the interval skips the step.

// The walk over the steps that one chunk of keys takes part in, the same for every wavefront of the workgroup.
struct SplitRingWalk {
    const Run *runs;
    const float *weights;
    int ri, rend;
    int W, kps, wg0, lon_lo, nkx, lat0, nlat, wlat0; // wlat0: quadrature weight of the run's latitude Run::pad is weights[pad + wlat0]
    // the run the walk stands in
    Run run;
    float w;
    int rl, par, vlo, nv, u0, m;
    // the step: band positions pos .. pos + HK of each wavefront's own 16 longitudes, up to `end`; rows [ua, ub) hold keys of the
    // chunk, vca = virtual column of row ua.  fresh: nothing of the band is staged yet
    int pos, end, ua, ub, vca;
    bool valid, fresh;
    __device__ inline void start(const Run *runs_, const float *weights_, int first, int rend_)
    {
        runs = runs_, weights = weights_, ri = first - 1, rend = rend_, m = 2, valid = false;
    }
    __device__ inline bool advance()
    {
        if (valid && pos + HK < end) {
            pos += HK;
            fresh = false;
            return true;
        }
        for (;;) {
            m++;
            if (m > 2) { // next run (a band of W + 63 rows on W >= 32 longitudes meets the chunk at most at m = -1 .. 2)
                ri++;
                if (ri >= rend) return valid = false;
                run = uniform_load(runs + ri);
                rl = run.pad - lat0; // row of the chunk
                m = 2;               // (skip the run unless the chunk holds part of it)
                if (rl < 0 || rl >= nlat) continue;
                par = 0, vlo = lon_lo, nv = nkx;
                if (kps > 1) {
                    par = run.lat - run.pad * kps; // column class: virtual column vc is real longitude vc * kps + par
                    vlo = (lon_lo - par + kps - 1) / kps;
                    nv = (lon_lo + nkx - par + kps - 1) / kps - vlo; // virtual columns vlo .. vlo + nv are in the chunk
                    if (nv <= 0) continue;
                }
                w = uniform_load(weights + (run.pad + wlat0));
                u0 = vlo - run.ws - wg0; // in (-2 W, W)
                u0 += (u0 < 0) ? W : 0;
                u0 += (u0 < 0) ? W : 0; // first band row at virtual column vlo
                m = -2;
                continue;
            }
            const int a0 = u0 + m * W, L = run.len + WQ - 1;
            const int a_ = max(a0, 0), b_ = min(a0 + nv, L);
            if (a_ >= b_) continue;
            ua = a_, ub = b_, vca = vlo + (a_ - a0);
            pos = max(0, ua - (WQ - HQ)), end = min(ub, run.len + HQ - 1);
            fresh = true;
            return valid = true;
        }
    }
};

// The walk of pass 2 over the scatter runs of one (virtual) input latitude: staged rows are queries, clipped to the local window.
// Row x of run (ws, len) of a workgroup at key column wg0 is (virtual) query column (wg0 - ws - len + 1 + x) mod W; the window
// holds the virtual columns 0 .. nv of the run's column class.
struct SplitRingWalk2 {
    const Run *runs;
    int ri, rend, W, wg0, qps, wo;
    Run run;
    int parq, nv, c0, u0, m;
    int pos, end, ua, ub, col; // as above; col = query column of row ua (whole: later rows wrap around)
    bool valid, fresh, whole;
    __device__ inline void start(const Run *runs_, int first, int rend_) { runs = runs_, ri = first - 1, rend = rend_, m = 2, valid = false; }
    __device__ inline bool advance()
    {
        if (valid && pos + HK < end) {
            pos += HK;
            fresh = false;
            return true;
        }
        for (;;) {
            m++;
            if (m > 2) { // next run
                ri++;
                if (ri >= rend) return valid = false;
                run = uniform_load(runs + ri);
                m = 2;
                parq = run.lat - run.pad * qps;
                nv = (wo - parq + qps - 1) / qps; // virtual columns of this class inside the window
                if (nv <= 0) continue;
                c0 = wg0 - run.ws - run.len + 1; // in (-2 W, W): query column of row 0
                c0 += (c0 < 0) ? W : 0;
                c0 += (c0 < 0) ? W : 0;
                whole = nv >= W;
                if (whole) { // the whole circle is local: one interval
                    ua = pos = 0, ub = run.len + WQ - 1, end = run.len + HQ - 1, col = c0;
                    fresh = true;
                    return valid = true;
                }
                u0 = c0 == 0 ? 0 : W - c0; // first row at column 0
                m = -2;
                continue;
            }
            const int a0 = u0 + m * W, L = run.len + WQ - 1;
            const int a_ = max(a0, 0), b_ = min(a0 + nv, L);
            if (a_ >= b_) continue;
            ua = a_, ub = b_, col = a_ - a0;
            pos = max(0, ua - (WQ - HQ)), end = min(ub, run.len + HQ - 1);
            fresh = true;
            return valid = true;
        }
    }
};

// Neighbors of a wavefront's column c that a step counts: element (kb, v) is neighbor t = tb + 16 kb + v, and it counts iff
// (unsigned)(t - lo) < n: 0 <= t < len and its row 16 wv + c + t lies in [ua, ub).  all: every element of every column does.
struct SplitRingMask {
    int tb, lo;
    unsigned n;
    bool all;
    __device__ inline SplitRingMask(int pos, int len, int ua, int ub, int wv, int c, int qd)
    {
        const int x0 = HQ * wv;
        tb = pos + 4 * qd - c;
        lo = max(0, ua - x0 - c);
        n = (unsigned)max(0, min(len, ub - x0 - c) - lo);
        all = pos >= HQ - 1 && pos + HK <= len && pos + x0 >= ua && pos + x0 + HK <= ub;
    }
    __device__ inline bool operator()(int kb, int v) const { return (unsigned)(tb + 16 * kb + v - lo) < n; }
};

// acc += x p, with the low-order products in a sum of their own or (one sum per block) added up first
template <int S> __device__ inline void s16_add(S16Sum &acc, const uint4 (&x)[3], const uint4 (&p)[3]) { s16_mma<S, 3>(acc, x, p); }
template <int S> __device__ inline void s16_add(f4v &acc, const uint4 (&x)[3], const uint4 (&p)[3])
{
    S16Sum t = {acc, f4v{0.f, 0.f, 0.f, 0.f}};
    s16_mma<S, 3>(t, x, p);
    acc = t.hi + t.lo;
}
__device__ inline void s16_set(S16Sum &s, f4v x) { s.hi = x, s.lo = f4v{0.f, 0.f, 0.f, 0.f}; }
__device__ inline void s16_set(f4v &s, f4v x) { s = x; }
__device__ inline void s16_rescale(S16Sum &s, float f) { s.hi *= f, s.lo *= f; }
__device__ inline void s16_rescale(f4v &s, float f) { s *= f; }

// MODE 0: the forward step.  MODE 1: pass 1, gather direction.  MODE 2: pass 1, up-sampling direction (see ring_m32_kernel, which
// states what each keeps and returns).  alpha_sum and qdotk_max of modes 0 and 1 come from the same operations in the same order.
template <typename T, int D, bool PAD, int MODE> __global__ __launch_bounds__(64 * NW, D <= 32 ? 3 : 2) void ring_s16_kernel(const Args a)
{
    constexpr bool PASS1 = MODE != 0, FIXED = MODE == 2;
    typedef SplitBand<T, D, PAD> Band_;
    constexpr int S = Band_::S, PITCH = Band_::PITCH, NCB = D / 16;
    extern __shared__ __attribute__((aligned(16))) char h16_lds[];
    char *Ks = h16_lds, *Vs = h16_lds + Band_::BYTES;

    S2_H16_IDS(a.Wo, a.Ho)
    (void)h, (void)nvalid; // heads are folded into the batch; the window can end before a class's last tile
    const int wv = __builtin_amdgcn_readfirstlane(wave);
    const int ho = a.gorder[a.row_first + rowsel]; // (virtual) output latitude
    const int hor = ho / a.r_qps, parq = ho - hor * a.r_qps;
    const int nclass = (a.r_wo - parq + a.r_qps - 1) / a.r_qps; // local queries of the virtual latitude
    if (wg0 >= nclass) return;
    const bool busy = active && w0 < nclass;
    const bool mine = busy && c < nclass - w0;
    const int n = PAD ? a.dk_ : D;
    const T *kx = static_cast<const T *>(a.k) + (size_t)b * a.r_nlat * a.r_nkx * n;
    const T *vx = static_cast<const T *>(a.v) + (size_t)b * a.r_nlat * a.r_nkx * n;
    const size_t pt = ((size_t)b * (a.Ho / a.r_qps) + hor) * a.r_wo + (size_t)(mine ? w0 + c : wg0) * a.r_qps + parq;

    { // the arc of columns this workgroup's queries can see, against the virtual columns that can lie in the chunk: most
      // workgroups of an equatorial latitude leave here, without reading a run
        typedef int i2v __attribute__((ext_vector_type(2)));
        const i2v span = uniform_load(reinterpret_cast<const i2v *>(a.gspan) + ho);
        const int la = span[1] + WQ - 1, b0 = a.r_lon_lo / a.kps, lb = (a.r_lon_lo + a.r_nkx - 1) / a.kps + 1 - b0;
        if (span[1] <= 0) return;
        if (la < a.Wi && lb < a.Wi) {
            int dab = (b0 - (wg0 + span[0])) % a.Wi; // chunk start relative to the arc's start
            dab += dab < 0 ? a.Wi : 0;
            if (dab >= la && a.Wi - dab >= lb) return;
        }
    }
    SplitRingWalk wk;
    wk.W = a.Wi, wk.kps = a.kps, wk.wg0 = wg0, wk.lon_lo = a.r_lon_lo, wk.nkx = a.r_nkx, wk.lat0 = a.r_lat0, wk.nlat = a.r_nlat, wk.wlat0 = a.r_wlat0;
    wk.start(a.gruns, a.quad_w, a.goff[ho], a.goff[ho + 1]);
    if (!wk.advance()) return; // nothing of this workgroup's neighborhood is in the chunk: the state stays as it is

    Band_ bd;
    const unsigned ldc = n * a.kps; // elements between two virtual columns
    auto fetch = [&]() __attribute__((always_inline)) {
        const int x0 = wk.fresh ? wk.pos : wk.pos + FRESH - HK; // band row of the first staged row
        const size_t base = ((size_t)wk.rl * a.r_nkx + (size_t)(wk.vca * a.kps + wk.par - a.r_lon_lo)) * n; // row ua
        if (wk.fresh)
            bd.template fetch_rows<FRESH>(kx + base, vx + base, tid, wk.ua - x0, wk.ub - x0, ldc, n);
        else
            bd.template fetch_rows<HK>(kx + base, vx + base, tid, wk.ua - x0, wk.ub - x0, ldc, n);
    };
    fetch();

    S16Own<T, D, false> qo, go;
    qo.template load<PAD>(static_cast<const T *>(a.q) + pt * n, n, qd);
    if constexpr (PASS1) go.template load<PAD>(static_cast<const T *>(a.dy) + pt * n, n, qd);
    // forward: Y^T; pass 1: alpha_k^T (acc) and alpha_kvw^T (acc2): register v of block cb is channel 16 cb + 4 qd + v of column c
    float *const acc_state = PASS1 ? a.r_ak : a.r_yacc;
    // (pass 1 of 64 channels has no registers for two sums per block)
    typedef typename std::conditional<PASS1 && (D > 32), f4v, S16Sum>::type Acc;
    Acc acc[NCB], acc2[PASS1 ? NCB : 1];
#pragma unroll
    for (int cb = 0; cb < NCB; cb++) {
        f4v x = {0.f, 0.f, 0.f, 0.f}, x2 = x;
        if (!PAD || 16 * cb + 4 * qd < n) {
            x = *reinterpret_cast<const f4v *>(acc_state + pt * n + 16 * cb + 4 * qd);
            if constexpr (PASS1) x2 = *reinterpret_cast<const f4v *>(a.r_akvw + pt * n + 16 * cb + 4 * qd);
        }
        s16_set(acc[cb], x);
        if constexpr (PASS1) s16_set(acc2[cb], x2);
    }
    // The exponentials are taken relative to a reference point m that is moved lazily; the exact maximum is kept per lane (mtrue)
    // and the sums are brought to it once, at the end.
    float m = fmaxf(a.r_qmax[pt], NEG_BIG_NAT), mtrue = -INFINITY;
    float Z = 0.f, I = 0.f; // the four lanes of a column each keep a share of the sums
    if constexpr (!FIXED) Z = qd == 0 ? a.r_asum[pt] : 0.f;
    if constexpr (PASS1) I = qd == 0 ? a.r_integral[pt] : 0.f;

    bd.template commit<FRESH>(Ks, Vs, tid, 0);
    __syncthreads();
    qo.settle_();
    if constexpr (PASS1) go.settle_();

    int rb = 0; // ring block of band position `pos`
    for (;;) {
        const float lw = fast_log2(wk.w);
        const int len = wk.run.len, pos = wk.pos, ua = wk.ua, ub = wk.ub;
        const bool more = wk.advance();
        if (more) fetch();

        const int x0 = pos + HQ * wv; // first row of this wavefront's step
        if (busy && x0 < ub && x0 + HK > ua) {
            const int b0 = s16_block(rb, wv), b1 = s16_block(b0, 1);
            const char *k0 = Ks + b0 * 16 * PITCH, *k1 = Ks + b1 * 16 * PITCH, *v0 = Vs + b0 * 16 * PITCH, *v1 = Vs + b1 * 16 * PITCH;
            f4v p[2], g[2];
            {
                S16Sum s[2] = {};
                s16_scores(s[0], k0, c, qd, qo);
                s16_scores(s[1], k1, c, qd, qo);
                p[0] = s16_value(s[0]), p[1] = s16_value(s[1]);
            }
            if constexpr (PASS1) {
                S16Sum s[2] = {};
                s16_scores(s[0], v0, c, qd, go);
                s16_scores(s[1], v1, c, qd, go);
                g[0] = s16_value(s[0]), g[1] = s16_value(s[1]);
            }
            const SplitRingMask counts(pos, len, ua, ub, wv, c, qd);
            if (!counts.all) {
#pragma unroll
                for (int kb = 0; kb < 2; kb++)
#pragma unroll
                    for (int v = 0; v < 4; v++) p[kb][v] = counts(kb, v) ? p[kb][v] : -INFINITY;
            }
            const float mx = fmaxf(fmaxf(fmaxf(p[0][0], p[0][1]), fmaxf(p[0][2], p[0][3])), fmaxf(fmaxf(p[1][0], p[1][1]), fmaxf(p[1][2], p[1][3])));
            if constexpr (!FIXED) mtrue = fmaxf(mtrue, mx);
            constexpr float THR = RESCALE_THR * 0.69314718f; // natural units
            if (!FIXED && __any(mx > m + THR)) {
                const float cm = h16_quarter_max(mx);
                const float mn = cm > m + THR ? cm : m; // m is finite, so mn is
                const float corr = fast_exp2((m - mn) * LOG2E);
                Z *= corr;
#pragma unroll
                for (int cb = 0; cb < NCB; cb++) s16_rescale(acc[cb], corr);
                if constexpr (PASS1) {
                    I *= corr;
#pragma unroll
                    for (int cb = 0; cb < NCB; cb++) s16_rescale(acc2[cb], corr);
                }
                m = mn;
            }
            const float sh = fmaf(-m, LOG2E, lw);
#pragma unroll
            for (int kb = 0; kb < 2; kb++) {
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    p[kb][v] = fast_exp2(fmaf(p[kb][v], LOG2E, sh)); // = exp(q.k - m) w; not counted: exp2(-inf) = 0
                    Z += p[kb][v];
                    if constexpr (PASS1) {
                        g[kb][v] *= p[kb][v]; // rows outside the chunk are staged as zeros, so <dy, v> is finite wherever p = 0
                        I += g[kb][v];
                    }
                }
            }
            uint4 ps[3], gs[3];
            s16_split_blocks(ps, p);
            if constexpr (PASS1) s16_split_blocks(gs, g);
            const char *r0 = PASS1 ? k0 : v0, *r1 = PASS1 ? k1 : v1;
#pragma unroll
            for (int cb = 0; cb < NCB; cb++) {
                uint4 x[3];
#pragma unroll
                for (int t = 0; t < S; t++) x[t] = h16_read_transposed<PITCH>(r0 + 2 * D * t, r1 + 2 * D * t, cb, c, qd);
                s16_add<S>(acc[cb], x, ps);
                if constexpr (PASS1) s16_add<S>(acc2[cb], x, gs);
            }
        }
        if (!more) break;
        __syncthreads(); // the next rows replace rows the slowest wavefront may still be reading
        rb = wk.fresh ? 0 : s16_block(rb, 2);
        if (wk.fresh)
            bd.template commit<FRESH>(Ks, Vs, tid, 0);
        else
            bd.template commit<HK>(Ks, Vs, tid, 16 * s16_block(rb, 3));
        __syncthreads();
    }

    Z = h16_quarter_sum(Z);
    if constexpr (PASS1) I = h16_quarter_sum(I);
    float f = 1.f;
    if constexpr (!FIXED) {
        mtrue = fmaxf(h16_quarter_max(mtrue), a.r_qmax[pt]); // the maximum over everything this column has seen, earlier chunks included (read again: a register less in the loop)
        f = mtrue > -INFINITY ? fast_exp2((m - mtrue) * LOG2E) : 1.f; // m <= mtrue <= m + THR; a column without neighbors keeps its zeros
    }
    if (mine) {
        if (qd == 0) {
            if constexpr (!FIXED) {
                a.r_asum[pt] = Z * f;
                a.r_qmax[pt] = mtrue;
            }
            if constexpr (PASS1) a.r_integral[pt] = I * f;
        }
#pragma unroll
        for (int cb = 0; cb < NCB; cb++) {
            if (!PAD || 16 * cb + 4 * qd < n) {
                *reinterpret_cast<f4v *>(acc_state + pt * n + 16 * cb + 4 * qd) = s16_value(acc[cb]) * f;
                if constexpr (PASS1) *reinterpret_cast<f4v *>(a.r_akvw + pt * n + 16 * cb + 4 * qd) = s16_value(acc2[cb]) * f;
            }
        }
    }
}

// Tiles of 64 virtual columns that hold any column class of a chunk of nkx longitudes
__host__ __device__ inline int ring_pass2_tiles(int nkx, int kps) { return (nkx / kps + WQ) / WQ; }

// Pass 2 (see ring_pass2_m32_kernel): dk, dv of the keys of one chunk.  A workgroup owns 64 consecutive virtual columns of one column
// class of a chunk latitude; every key belongs to one wavefront, so dk, dv are added to (WRITE: written) plainly.
template <typename T, int D, bool PAD, bool WRITE> __global__ __launch_bounds__(64 * NW, D <= 32 ? 3 : 2) void ring_pass2_s16_kernel(const Args a)
{
    typedef SplitBand<T, D, PAD> Band_;
    constexpr int S = Band_::S, PITCH = Band_::PITCH, NCB = D / 16;
    extern __shared__ __attribute__((aligned(16))) char h16_lds[];
    char *Qs = h16_lds, *Gs = h16_lds + Band_::BYTES;
    float2 *Ts = reinterpret_cast<float2 *>(h16_lds + 2 * Band_::BYTES); // (log2 w - log2 sum alpha, -integral_norm) of the staged queries
    const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, qd = lane >> 4;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = PAD ? a.dk_ : D;
    // workgroup -> (batch, virtual input latitude in the plan's order, tile of 64 virtual columns of the chunk)
    const int ntile = ring_pass2_tiles(a.r_nkx, a.kps);
    int id = blockIdx.x;
    const int b = id % a.B;
    id /= a.B;
    const int hv = a.sorder[id / ntile], tile = id % ntile;
    const int hreal = hv / a.kps, par = hv - hreal * a.kps, rl = hreal - a.r_lat0;
    if (rl < 0 || rl >= a.r_nlat) return;
    const int vlo = (a.r_lon_lo - par + a.kps - 1) / a.kps, nv = (a.r_lon_lo + a.r_nkx - par + a.kps - 1) / a.kps - vlo;
    if (WQ * tile >= nv) return;
    const int wg0 = vlo + WQ * tile; // first virtual column of the workgroup
    const int left = nv - WQ * tile - HQ * wv; // columns from this wavefront's first one on
    const bool busy = left > 0, mine = c < left;
    const size_t pt = ((size_t)b * a.r_nlat + rl) * a.r_nkx + (size_t)((wg0 + (mine ? HQ * wv + c : 0)) * a.kps + par - a.r_lon_lo); // the key in the chunk

    SplitRingWalk2 wk;
    wk.W = a.Wi, wk.wg0 = wg0, wk.qps = a.r_qps, wk.wo = a.r_wo;
    wk.start(a.sruns, a.soff[hv], a.soff[hv + 1]);
    const bool any = (WRITE || ring_window_seen(a.sruns, a.soff[hv], a.soff[hv + 1], lane, wg0, WQ, a.Wi, a.r_qps, a.r_wo)) && wk.advance(); // false: none of the queries that see these keys is local
    if (!WRITE && !any) return;

    const size_t sbase = (size_t)b * (a.Ho / a.r_qps) * a.r_wo; // first local query of the batch entry
    const T *qy = static_cast<const T *>(a.q) + sbase * n;
    const T *gy = static_cast<const T *>(a.dy) + sbase * n;
    S16Own<T, D, false> ko, vo;
    ko.template load<PAD>(static_cast<const T *>(a.k) + pt * n, n, qd);
    vo.template load<PAD>(static_cast<const T *>(a.v) + pt * n, n, qd);
    f4v dkt[NCB], dvt[NCB];
    s16_zero(dkt);
    s16_zero(dvt);
    const float lw = fast_log2(a.quad_w[hreal + a.r_wlat0]);

    Band_ bd;
    float st_a = 0.f, st_m = 0.f, st_i = 0.f; // alpha_sum, qdotk_max, integral_norm of a staged row, as loaded: first used in commit
    const unsigned ldc = n * a.r_qps; // elements between two virtual query columns
    auto fetch = [&]() __attribute__((always_inline)) {
        const int x0 = wk.fresh ? wk.pos : wk.pos + FRESH - HK, rows = wk.fresh ? FRESH : HK;
        // the run's output latitude is virtual (real latitude Run::pad, column class parq): virtual column j is the local query
        // column j * r_qps + parq
        const size_t lat = (size_t)wk.run.pad * a.r_wo + wk.parq;
        const int wrap = wk.whole ? wk.W : 0;
        const int lo = wk.ua - x0, hi = wk.ub - x0;
        if (wk.fresh)
            bd.template fetch_rows<FRESH>(qy + lat * n, gy + lat * n, tid, lo, hi, ldc, n, wk.col, wrap);
        else
            bd.template fetch_rows<HK>(qy + lat * n, gy + lat * n, tid, lo, hi, ldc, n, wk.col, wrap);
        if (tid < rows) { // the first threads fetch the statistics of the staged rows
            st_a = 0.f;
            if (tid >= lo && tid < hi) {
                int col = wk.col + tid - lo;
                while (wrap && col >= wrap) col -= wrap;
                const size_t s = sbase + lat + (size_t)col * a.r_qps;
                st_a = a.r_asum[s], st_m = a.r_qmax[s], st_i = a.r_integral[s];
            }
        }
    };
    auto commit = [&](bool fresh, int x0) __attribute__((always_inline)) {
        if (fresh)
            bd.template commit<FRESH>(Qs, Gs, tid, 0);
        else
            bd.template commit<HK>(Qs, Gs, tid, x0);
        if (tid < (fresh ? FRESH : HK)) {
            int r = x0 + tid;
            r -= r >= FRESH ? FRESH : 0;
            // (a query that saw nothing, or a row outside the window: a probability of exp2(-inf) = 0)
            Ts[r] = st_a > 0.f ? make_float2(lw - fmaf(st_m, LOG2E, fast_log2(st_a)), -st_i) : make_float2(-INFINITY, 0.f);
        }
    };
    if (any) {
        fetch();
        commit(true, 0);
    }
    __syncthreads();
    ko.settle_();
    vo.settle_();

    int rb = 0;
    bool more = any;
    while (more) {
        const int len = wk.run.len, pos = wk.pos, ua = wk.ua, ub = wk.ub;
        more = wk.advance();
        if (more) fetch();

        const int x0 = pos + HQ * wv;
        if (busy && x0 < ub && x0 + HK > ua) {
            const int blk[2] = {s16_block(rb, wv), s16_block(s16_block(rb, wv), 1)};
            const char *q0 = Qs + blk[0] * 16 * PITCH, *q1 = Qs + blk[1] * 16 * PITCH, *g0 = Gs + blk[0] * 16 * PITCH, *g1 = Gs + blk[1] * 16 * PITCH;
            S16Sum sc[2] = {}, gc[2] = {};
            f4v lv[2];
#pragma unroll
            for (int qb = 0; qb < 2; qb++) { // the products with dy start at -integral_norm
                const float4 *sp = reinterpret_cast<const float4 *>(Ts + 16 * blk[qb] + 4 * qd);
                const float4 s01 = sp[0], s23 = sp[1];
                lv[qb] = f4v{s01.x, s01.z, s23.x, s23.z};
                gc[qb].hi = f4v{s01.y, s01.w, s23.y, s23.w};
            }
            s16_scores(sc[0], q0, c, qd, ko);
            s16_scores(sc[1], q1, c, qd, ko);
            s16_scores(gc[0], g0, c, qd, vo);
            s16_scores(gc[1], g1, c, qd, vo);
            const SplitRingMask counts(pos, len, ua, ub, wv, c, qd);
            f4v p[2], ds[2];
#pragma unroll
            for (int qb = 0; qb < 2; qb++) {
                const f4v s = s16_value(sc[qb]), g = s16_value(gc[qb]);
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    p[qb][v] = fast_exp2(fmaf(s[v], LOG2E, lv[qb][v])); // = alpha / alpha_sum
                    if (!counts.all) p[qb][v] = counts(qb, v) ? p[qb][v] : 0.f;
                    ds[qb][v] = p[qb][v] * g[v];
                }
            }
            uint4 ps[3];
            s16_split_blocks(ps, p);
            s16_accumulate<D, S>(dvt, g0, g1, c, qd, ps);
            s16_split_blocks(ps, ds);
            s16_accumulate<D, S>(dkt, q0, q1, c, qd, ps);
        }
        if (!more) break;
        __syncthreads();
        rb = wk.fresh ? 0 : s16_block(rb, 2);
        commit(wk.fresh, wk.fresh ? 0 : 16 * s16_block(rb, 3));
        __syncthreads();
    }

    if (mine) {
        float *dk = static_cast<float *>(a.dk) + pt * n + 4 * qd, *dv = static_cast<float *>(a.dv) + pt * n + 4 * qd;
#pragma unroll
        for (int cb = 0; cb < NCB; cb++) {
            if (!PAD || 16 * cb + 4 * qd < n) {
                f4v x = s16_value(dkt[cb]), y = s16_value(dvt[cb]);
                if (!WRITE) x += *reinterpret_cast<const f4v *>(dk + 16 * cb), y += *reinterpret_cast<const f4v *>(dv + 16 * cb);
                *reinterpret_cast<f4v *>(dk + 16 * cb) = x;
                *reinterpret_cast<f4v *>(dv + 16 * cb) = y;
            }
        }
    }
}
