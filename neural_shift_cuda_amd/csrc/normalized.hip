// normalized.hip -- overflow-safe normalized accumulation D = K/C on gfx950.
//
// Semantics (reference GPU kernels csrc/shift_ops_cuda.cu:474-791):
//   terms i of pixel p: forward (w_s[p], x[(p+s) mod]) and, for has_inv rows
//   with box(p-s), mirror (w_s[p-s], x[p-s]).  Keys are the positive weights
//   (log_weights = 0) or the logits (log_weights = 1); w == 0 / l == -inf are
//   masks.  D = sum a_i v_i / sum a_i with a_i = w_i / max w or
//   exp(l_i - max l); log_C = log(max w) + log(sum a) or max l + log(sum a).
//   Empty rows give D = 0, log_C = -inf; a NaN / +inf key, or a negative
//   positive weight, gives NaN in both outputs.
//
// Forward: a single pass over the weight planes as an online softmax.  Each
// lane keeps (m, u, z) per pixel; a term with key k updates
//   k > m : u = u*r + v, z = z*r + 1, m = k      with r = rescale(m -> k)
//   k <= m: u += a v,    z += a                  with a = scale(k -> m)
// where both branches share one transcendental (log mode: exp(-|k - m|)) or
// one division (positive mode: min(k, m) / max(k, m)), so every term costs
// one exp or one divide and the weights are read from HBM exactly once.
//
// Backward (csrc/shift_ops_cuda.cu:655-791), one fused pass per tile:
//   f(v, L) = 0 if lw(v) == -inf or L == -inf else exp(lw(v) - L)
//   gx[q]   = sum_s f(w_s[o], L[o]) gD[o] at o = (q-s) mod
//           + [inv, box(q+s)] f(w_s[q], L[q+s]) gD[q+s]
//   gw_s[q] = 0 for a masked weight, else
//             F(L[q]) score(q, x[(q+s) mod]) + [inv, box(q+s)] F(L[q+s]) score(q+s, x[q])
//   score(o, v) = gD[o] (v - D[o]) + gLogC[o];  F = f (log mode) or exp(-L).
#include <algorithm>
#include <cstdlib>
#include <initializer_list>
#include <type_traits>

#include "nsh_common.hpp"
#include "scatter.hpp"

namespace nsh {

template <int VEC>
struct NGeo {
    static constexpr int TW = kTPR * VEC;
    static constexpr int TH = kRows;
    static constexpr int LW = TW + 2 * kRmax;
    static constexpr int LH = TH + 2 * kRmax;
};

template <typename A> struct Lim;
template <> struct Lim<float> {
    static __device__ __forceinline__ float maxv() { return 3.4028234663852886e38f; }
    static __device__ __forceinline__ float inf() { return __builtin_inff(); }
    static __device__ __forceinline__ float nan() { return __builtin_nanf(""); }
    static __device__ __forceinline__ float ex(float v) { return ::expf(v); }
    static __device__ __forceinline__ float lg(float v) { return ::logf(v); }
};
template <> struct Lim<double> {
    static __device__ __forceinline__ double maxv() { return 1.7976931348623157e308; }
    static __device__ __forceinline__ double inf() { return __builtin_inf(); }
    static __device__ __forceinline__ double nan() { return __builtin_nan(""); }
    static __device__ __forceinline__ double ex(double v) { return ::exp(v); }
    static __device__ __forceinline__ double lg(double v) { return ::log(v); }
};

// Per-pixel online-softmax state.
template <typename A>
struct Online {
    A m, u, z;
    bool any, bad;
};

template <typename A, bool LOGW>
__device__ __forceinline__ void online_init(Online<A>& st) {
    st.m = LOGW ? -Lim<A>::maxv() : A(0);
    st.u = A(0);
    st.z = A(0);
    st.any = false;
    st.bad = false;
}

// Masked key: a term that changes no state.
template <typename A, bool LOGW>
__device__ __forceinline__ A masked_key() {
    return LOGW ? -Lim<A>::inf() : A(0);
}

template <typename A, bool LOGW>
__device__ __forceinline__ void online_add(Online<A>& st, A k, A v) {
    bool valid;
    A r, a;
    bool gt;
    if (LOGW) {
        valid = k > -Lim<A>::inf() && k <= Lim<A>::maxv();
        st.bad |= (k != k) || (k > Lim<A>::maxv());  // NaN or +inf
        const A d = k - st.m;
        gt = d > A(0);
        const A t = Lim<A>::ex(-__builtin_fabs(d));
        r = gt ? t : A(1);
        a = gt ? A(1) : t;
    } else {
        valid = k > A(0) && k <= Lim<A>::maxv();
        st.bad |= !(k >= A(0)) || k > Lim<A>::maxv();  // negative, NaN or +inf
        gt = k > st.m;
        const A num = gt ? st.m : k;
        const A den = gt ? k : st.m;
        const A t = num / den;
        r = gt ? t : A(1);
        a = gt ? A(1) : t;
    }
    r = valid ? r : A(1);
    a = valid ? a : A(0);
    st.u = fma_acc(st.u, r, a * v);
    st.z = fma_acc(st.z, r, a);
    st.m = (valid && gt) ? k : st.m;
    st.any |= valid;
}

template <typename A, bool LOGW>
__device__ __forceinline__ void online_final(const Online<A>& st, A& D, A& L) {
    if (st.bad) {
        D = Lim<A>::nan();
        L = Lim<A>::nan();
    } else if (!st.any) {
        D = A(0);
        L = -Lim<A>::inf();
    } else {
        D = st.u / st.z;
        L = (LOGW ? st.m : Lim<A>::lg(st.m)) + Lim<A>::lg(st.z);
    }
}

// A weight that breaks the op's contract: a NaN or +inf logit; a negative,
// NaN or +inf positive weight.  The kernels' states already carry every such
// key they take in (NaN in both outputs), so a forward asked to check the
// weights (weights_ok) reads the answer off its states and tests a weight
// itself only where the forward box drops it; a separate pass over the
// weights is not needed (c3 positive, 1.5 GB of fp32 weights: the check took
// 2.2 ms as elementwise passes, and the whole forward takes 0.30 ms with or
// without it).
template <typename A, bool LOGW>
__device__ __forceinline__ bool key_bad(A k) {
    return LOGW ? !(k <= Lim<A>::maxv()) : !(k >= A(0) && k <= Lim<A>::maxv());
}

__device__ __forceinline__ bool tile_inside_n(int h0, int w0, int TH, int TW, int H, int W, int dx,
                                              int dy) {
    const int h1 = (h0 + TH < H ? h0 + TH : H) - 1;
    const int w1 = (w0 + TW < W ? w0 + TW : W) - 1;
    return h0 + dx >= 0 && h1 + dx < H && w0 + dy >= 0 && w1 + dy < W;
}

template <typename T, int VEC, bool LOGW>
__global__ __launch_bounds__(kThreads) void normalized_fwd_kernel(
    const T* __restrict__ x, const T* __restrict__ w, const int64_t* __restrict__ shifts, int S,
    int codes, int C, int H, int W, int ntw, int nth, int64_t plane_step,
    acc_t<T>* __restrict__ Dout, acc_t<T>* __restrict__ Lout, int* __restrict__ weights_ok) {
    using A = acc_t<T>;
    using G = NGeo<VEC>;
    extern __shared__ __align__(16) unsigned char smem[];
    int4* shl = reinterpret_cast<int4*>(smem);
    A* xt = reinterpret_cast<A*>(smem + shift_lds_bytes(S));

    const TileIdx ti = tile_of(xcd_tile(blockIdx.x, gridDim.x), ntw, nth, G::TH, G::TW);
    const int64_t HW = static_cast<int64_t>(H) * W;
    const T* xp = x + ti.bc * HW;
    stage_shifts(shl, shifts, S, 3, H, W, codes);
    stage_tile<T, A>(xt, xp, H, W, ti.h0, ti.w0, G::LH, G::LW);
    __syncthreads();

    const int tx = threadIdx.x % kTPR;
    const int ty = threadIdx.x / kTPR;
    const int h = ti.h0 + ty;
    const int w0 = ti.w0 + tx * VEC;
    if (h >= H || w0 >= W) return;
    const uint32_t own = static_cast<uint32_t>(h) * static_cast<uint32_t>(W) + w0;
    const int lc = (ty + kRmax) * G::LW + tx * VEC + kRmax;
    const int64_t b = ti.bc / C;
    const int64_t c = ti.bc - b * C;
    const bool wsh = (codes & kCodesSharedW) != 0;
    const T* wp = w + weight_plane(b, c, C, wsh) * HW;
    const int64_t wstep = weight_step(plane_step, C, wsh);

    Online<A> st[VEC];
#pragma unroll
    for (int k = 0; k < VEC; ++k) online_init<A, LOGW>(st[k]);
    bool bad = false;  // a weight outside the contract (weights_ok)

    for (int s = 0; s < S; ++s, wp += wstep) {
        const ShiftRec r = read_shift(shl, s);
        const bool lds = shift_in_lds(r);
        A wv[VEC], xv[VEC];
        load_acc<T, VEC>(wp + own, wv);
        if (lds) {
            const A* xr = xt + lc + r.dx * G::LW + r.dy;
#pragma unroll
            for (int k = 0; k < VEC; ++k) xv[k] = xr[k];
        } else {
            int hh = h + r.dxm;
            hh -= hh >= H ? H : 0;
#pragma unroll
            for (int k = 0; k < VEC; ++k) {
                int ww = w0 + k + r.dym;
                ww -= ww >= W ? W : 0;
                xv[k] = to_acc(xp[static_cast<uint32_t>(hh) * W + ww]);
            }
        }
#pragma unroll
        for (int k = 0; k < VEC; ++k) {
            if (weights_ok != nullptr) bad |= key_bad<A, LOGW>(wv[k]);
            online_add<A, LOGW>(st[k], fwd_kept(r, h, w0 + k, H, W) ? wv[k]
                                                                    : masked_key<A, LOGW>(),
                                xv[k]);
        }

        if (r.inv) {
            // source (h - dx, w - dy), wrapped for a circular mirror
            const bool rok = r.per || in_range(h - r.dx, H);
            int hs = h - r.dxm;
            hs += hs < 0 ? H : 0;
#pragma unroll
            for (int k = 0; k < VEC; ++k) {
                if (rok && (r.per || in_range(w0 + k - r.dy, W))) {
                    int ws = w0 + k - r.dym;
                    ws += ws < 0 ? W : 0;
                    const uint32_t src = static_cast<uint32_t>(hs) * W + ws;
                    const A wi = to_acc(wp[src]);
                    const A xi = lds ? xt[lc - r.dx * G::LW - r.dy + k] : to_acc(xp[src]);
                    online_add<A, LOGW>(st[k], wi, xi);
                }
            }
        }
    }
    if (weights_ok != nullptr && bad) *weights_ok = 0;
    A Dv[VEC], Lv[VEC];
#pragma unroll
    for (int k = 0; k < VEC; ++k) online_final<A, LOGW>(st[k], Dv[k], Lv[k]);
    store_out<A, VEC>(Dout + ti.bc * HW + own, Dv);
    store_out<A, VEC>(Lout + ti.bc * HW + own, Lv);
}

// lw(v): the log-weight of a key (positive mode: log v, -inf for 0, NaN < 0).
template <typename A, bool LOGW>
__device__ __forceinline__ A as_log(A v) {
    if (LOGW) return v;
    return v > A(0) ? Lim<A>::lg(v) : (v == A(0) ? -Lim<A>::inf() : Lim<A>::nan());
}

template <typename A>
__device__ __forceinline__ A frac(A lw, A L) {
    return (lw == -Lim<A>::inf() || L == -Lim<A>::inf()) ? A(0) : Lim<A>::ex(lw - L);
}

template <typename T, int VEC, bool LOGW>
__global__ __launch_bounds__(kThreads) void normalized_bwd_kernel(
    const T* __restrict__ x, const T* __restrict__ w, const acc_t<T>* __restrict__ Dg,
    const acc_t<T>* __restrict__ Lg, const acc_t<T>* __restrict__ gDg,
    const acc_t<T>* __restrict__ gLg, const int64_t* __restrict__ shifts, int S, int codes, int C,
    int H, int W, int ntw, int nth, int64_t plane_step, T* __restrict__ gx, T* __restrict__ gw) {
    using A = acc_t<T>;
    using G = NGeo<VEC>;
    constexpr int LT = G::LH * G::LW;
    extern __shared__ __align__(16) unsigned char smem[];
    int4* shl = reinterpret_cast<int4*>(smem);
    A* xt = reinterpret_cast<A*>(smem + shift_lds_bytes(S));
    A* dt = xt + LT;
    A* lt = dt + LT;
    A* gdt = lt + LT;
    A* glt = gdt + LT;

    const TileIdx ti = tile_of(xcd_tile(blockIdx.x, gridDim.x), ntw, nth, G::TH, G::TW);
    const int64_t HW = static_cast<int64_t>(H) * W;
    const T* xp = x + ti.bc * HW;
    const A* Dp = Dg + ti.bc * HW;
    const A* Lp = Lg + ti.bc * HW;
    const A* gDp = gDg + ti.bc * HW;
    const A* gLp = gLg + ti.bc * HW;
    stage_shifts(shl, shifts, S, 3, H, W, codes);
    stage_tile<T, A>(xt, xp, H, W, ti.h0, ti.w0, G::LH, G::LW);
    stage_tile_acc<A>(dt, Dp, H, W, ti.h0, ti.w0, G::LH, G::LW);
    stage_tile_acc<A>(lt, Lp, H, W, ti.h0, ti.w0, G::LH, G::LW);
    stage_tile_acc<A>(gdt, gDp, H, W, ti.h0, ti.w0, G::LH, G::LW);
    stage_tile_acc<A>(glt, gLp, H, W, ti.h0, ti.w0, G::LH, G::LW);
    __syncthreads();

    const int tx = threadIdx.x % kTPR;
    const int ty = threadIdx.x / kTPR;
    const int h = ti.h0 + ty;
    const int w0 = ti.w0 + tx * VEC;
    if (h >= H || w0 >= W) return;
    const uint32_t own = static_cast<uint32_t>(h) * static_cast<uint32_t>(W) + w0;
    const int lc = (ty + kRmax) * G::LW + tx * VEC + kRmax;
    const int64_t b = ti.bc / C;
    const int64_t c = ti.bc - b * C;
    const bool wsh = (codes & kCodesSharedW) != 0;
    const T* wp = w + weight_plane(b, c, C, wsh) * HW;
    const int64_t wstep = weight_step(plane_step, C, wsh);
    T* gp = gw + (b * C + c) * HW;  // the gradient has every channel

    A xo[VEC], Do[VEC], Lo[VEC], gDo[VEC], gLo[VEC], Eo[VEC], gxa[VEC];
#pragma unroll
    for (int k = 0; k < VEC; ++k) {
        xo[k] = xt[lc + k];
        Do[k] = dt[lc + k];
        Lo[k] = lt[lc + k];
        gDo[k] = gdt[lc + k];
        gLo[k] = glt[lc + k];
        Eo[k] = Lim<A>::ex(-Lo[k]);
        gxa[k] = A(0);
    }

    for (int s = 0; s < S; ++s, wp += wstep, gp += plane_step) {
        const ShiftRec r = read_shift(shl, s);
        const bool lds = shift_in_lds(r);
        // neighbour values at q + s (circular) and q - s (circular)
        A xf[VEC], Dp_[VEC], Lp_[VEC], gDp_[VEC], gLp_[VEC], Lm[VEC], gDm[VEC];
        if (lds) {
            const int op = lc + r.dx * G::LW + r.dy;
            const int om = lc - r.dx * G::LW - r.dy;
#pragma unroll
            for (int k = 0; k < VEC; ++k) {
                xf[k] = xt[op + k];
                Dp_[k] = dt[op + k];
                Lp_[k] = lt[op + k];
                gDp_[k] = gdt[op + k];
                gLp_[k] = glt[op + k];
                Lm[k] = lt[om + k];
                gDm[k] = gdt[om + k];
            }
        } else {
            int hp = h + r.dxm;
            hp -= hp >= H ? H : 0;
            int hm = h - r.dxm;
            hm += hm < 0 ? H : 0;
#pragma unroll
            for (int k = 0; k < VEC; ++k) {
                int wq = w0 + k + r.dym;
                wq -= wq >= W ? W : 0;
                int wm = w0 + k - r.dym;
                wm += wm < 0 ? W : 0;
                const uint32_t ip = static_cast<uint32_t>(hp) * W + wq;
                const uint32_t im = static_cast<uint32_t>(hm) * W + wm;
                xf[k] = to_acc(xp[ip]);
                Dp_[k] = Dp[ip];
                Lp_[k] = Lp[ip];
                gDp_[k] = gDp[ip];
                gLp_[k] = gLp[ip];
                Lm[k] = Lp[im];
                gDm[k] = gDp[im];
            }
        }
        bool okp[VEC];
        {
            const bool rok = r.per || in_range(h + r.dx, H);
#pragma unroll
            for (int k = 0; k < VEC; ++k)
                okp[k] = r.inv && rok && (r.per || in_range(w0 + k + r.dy, W));
        }

        A wv[VEC];
        load_acc<T, VEC>(wp + own, wv);
        A g[VEC];
#pragma unroll
        for (int k = 0; k < VEC; ++k) {
            // forward box: a dropped w_s[q] acts as a masked key
            const A lw = fwd_kept(r, h, w0 + k, H, W) ? as_log<A, LOGW>(wv[k]) : -Lim<A>::inf();
            A Fi = A(0), si = A(0);
            if (okp[k]) {
                si = fma_acc(gDp_[k], xo[k] - Dp_[k], gLp_[k]);
                Fi = LOGW ? frac<A>(lw, Lp_[k]) : Lim<A>::ex(-Lp_[k]);
                // gx mirror term: f(w_s[q], L[q+s]) gD[q+s]
                gxa[k] = fma_acc(frac<A>(lw, Lp_[k]), gDp_[k], gxa[k]);
            }
            const A sf = fma_acc(gDo[k], xf[k] - Do[k], gLo[k]);
            const A Ff = LOGW ? frac<A>(lw, Lo[k]) : Eo[k];
            const A gv = fma_acc(Ff, sf, Fi * si);
            g[k] = (lw == -Lim<A>::inf()) ? A(0) : gv;
        }
        store_acc<T, VEC>(gp + own, g, true);

        // gx forward term at o = (q - s) mod
        A ws[VEC];
        if (tile_inside_n(ti.h0, ti.w0, G::TH, G::TW, H, W, -r.dx, -r.dy)) {
            const int off = -(r.dx * W + r.dy);
#pragma unroll
            for (int k = 0; k < VEC; ++k) ws[k] = to_acc(wp[static_cast<int64_t>(own) + off + k]);
        } else {
            int hm = h - r.dxm;
            hm += hm < 0 ? H : 0;
#pragma unroll
            for (int k = 0; k < VEC; ++k) {
                int wm = w0 + k - r.dym;
                wm += wm < 0 ? W : 0;
                ws[k] = to_acc(wp[static_cast<uint32_t>(hm) * W + wm]);
            }
        }
#pragma unroll
        for (int k = 0; k < VEC; ++k) {
            const A lw = fwd_kept_src(r, h, w0 + k, H, W) ? as_log<A, LOGW>(ws[k]) : -Lim<A>::inf();
            gxa[k] = fma_acc(frac<A>(lw, Lm[k]), gDm[k], gxa[k]);
        }
    }
    store_acc<T, VEC>(gx + ti.bc * HW + own, gxa, false);
}

// ---------------------------------------------------------------------------
// Scatter form: every weight element is read once, aligned.
//
// The kernels above gather the mirror term of pixel p from w_s[p - s] (and,
// in the backward, the x-gradient term from w_s[(q - s) mod]): reads R rows /
// columns into the neighbouring tile, mostly missed in L2.  The scatter
// kernels below use the lane owning q, which holds w_s[q], for every term
// that weight enters:
//   forward : the mirror term (w_s[q], x[q]) of p = q + s is merged into an
//             LDS window of online-softmax states (m, u, z) at q + s.  The
//             merge of two states is associative, so the window, its border
//             spilled to the workspace, and the lane's own register state
//             combine in any fixed order; normalized_fixup_kernel merges the
//             neighbours' spills into the pixels near a tile edge (whose
//             partial states the main kernel leaves in the workspace) and
//             finishes D and log_C.  A state carries "no valid term" as
//             z == 0 and "bad key" as z = NaN.
//   backward: f(w_s[q], L[q]) gD[q], the x-gradient term of q + s, is added
//             into an LDS window at q + s (circular), as accumulate_uz's
//             backward does; spill_fixup_kernel adds the window borders.
//             Positive weights use E = exp(-L) staged per pixel:
//             f(w, L) = w E, so no transcendental per term.
// Shifts beyond the LDS halo take the gather form in a second loop, so the
// prefetch ring loop issues no conditional loads.  Lane ownership is
// strided (SGeo): LDS accesses are free of bank conflicts.
// ---------------------------------------------------------------------------

// Per-term arithmetic of the scatter kernels.  fp32 uses the hardware exp2
// (v_exp_f32) on x log2(e); its relative error grows like |x| 2^-24, which
// only matters for terms below exp(-87) that fp32 flushes anyway.  fp64
// keeps the library exp.
template <typename A> struct NMath;
template <> struct NMath<float> {
    static __device__ __forceinline__ float ex(float v) {
        return __builtin_amdgcn_exp2f(v * 1.44269504088896341f);
    }
    static __device__ __forceinline__ int fexp(float v) { return __builtin_amdgcn_frexp_expf(v); }
    static __device__ __forceinline__ float ldx(float v, int e) {
        return __builtin_amdgcn_ldexpf(v, e);
    }
};
template <> struct NMath<double> {
    static __device__ __forceinline__ double ex(double v) { return ::exp(v); }
    static __device__ __forceinline__ int fexp(double v) { return __builtin_amdgcn_frexp_exp(v); }
    static __device__ __forceinline__ double ldx(double v, int e) {
        return __builtin_amdgcn_ldexp(v, e);
    }
};

// Online-softmax state (m, u, z): u = sum a_i v_i and z = sum a_i over the
// terms seen so far, with a_i = exp(l_i - m), m the largest logit (log
// weights), or a_i = w_i 2^-m, m the binary exponent of the largest weight
// (positive weights: power-of-two scaling is exact and needs no divide; the
// largest term has a >= 1/2, so z cannot overflow).  z == 0: no valid
// term; z = NaN: a bad key (NaN / +inf logit; negative, NaN or +inf weight).
// Initial state: (empty_m, 0, 0).
template <typename A, bool LOGW>
__device__ __forceinline__ A empty_m() {
    // below every binary exponent of a nonzero value (fp32 >= -148, fp64 >= -1073)
    return LOGW ? -Lim<A>::maxv() : A(sizeof(A) == 8 ? -2000 : -1000);
}

template <typename A, bool LOGW>
__device__ __forceinline__ void term_add(A& m, A& u, A& z, A k, A v) {
    using M = NMath<A>;
    if (LOGW) {
        // -inf (mask) changes nothing below.  A NaN key makes a and hence u
        // and z NaN.  A +inf key (bad) sets m = +inf: every later key or
        // merge then forms exp(inf - inf) = NaN, and state_final reports a
        // state still at m = +inf as NaN, so no per-term test is needed.
        const A d = k - m;
        const bool gt = d > A(0);
        const A t = M::ex(-__builtin_fabs(d));
        const A r = gt ? t : A(1);
        const A a = gt ? A(1) : t;
        u = fma_acc(u, r, a * v);
        z = fma_acc(z, r, a);
        m = gt ? k : m;
    } else {
        const bool bad = !(k >= A(0)) || k > Lim<A>::maxv();
        const int me = static_cast<int>(m);
        const int e = k > A(0) ? M::fexp(k) : static_cast<int>(empty_m<A, false>());
        const int dd = me - e < 0 ? me - e : 0;  // rescale when the maximum grows
        const int mn = me > e ? me : e;
        const A a = M::ldx(k, -mn);
        u = fma_acc(a, v, M::ldx(u, dd));
        z = M::ldx(z, dd) + a;
        z = bad ? Lim<A>::nan() : z;
        m = static_cast<A>(mn);
    }
}

// term_add with a lazy reference point.  m need not be the largest key: a
// term may weigh up to e^kLazyLog (log weights) or 2^kLazyExp (positive
// weights) relative to m, and m moves (u and z rescaled) only when a key
// exceeds that, in practice at a state's first term.  The common term is
// then one exp (or one ldexp), one compare and two adds, and the rare one
// takes a branch that a wave skips when none of its lanes needs it.  Any
// (m, u, z) with a = weight relative to m is a valid state for term_add,
// state_merge and state_final, so the two forms mix freely.  Range: u and z
// stay below 2^11 (at most 2048 terms) times e^16 resp. 2^24 (times max |v|
// for u), far inside the accumulator range for image values.
constexpr float kLazyLog = 16.0f;
constexpr int kLazyExp = 24;

template <typename A>
__device__ __forceinline__ bool below_lazy_bound(A a) {
    // a in [+0, 2^kLazyExp): one unsigned compare of the bit pattern (a
    // negative value, -0, NaN and +inf all compare above the bound)
    if constexpr (sizeof(A) == 4)
        return __float_as_uint(a) < __float_as_uint(static_cast<float>(1 << kLazyExp));
    else
        return static_cast<uint64_t>(__double_as_longlong(a)) <
               static_cast<uint64_t>(__double_as_longlong(static_cast<double>(1 << kLazyExp)));
}

template <typename A, bool LOGW>
__device__ __forceinline__ void term_add_lazy(A& m, A& u, A& z, A k, A v) {
    using M = NMath<A>;
    if (LOGW) {
        // k - m > bound: move m to k (also for a +inf key, whose a is then
        // exp(inf - inf) = NaN: bad).  A NaN key gives a = NaN, a -inf
        // (masked) key a = 0.  The empty state (m = -maxv) takes the branch
        // with any finite key and rescales its zeros.
        if (__builtin_expect(k - m > A(kLazyLog), 0)) {
            const A r = M::ex(m - k);
            u *= r;
            z *= r;
            m = k;
        }
        const A a = M::ex(k - m);
        u = fma_acc(a, v, u);
        z += a;
    } else {
        const A a = M::ldx(k, -static_cast<int>(m));
        if (__builtin_expect(below_lazy_bound(a), 1)) {
            u = fma_acc(a, v, u);
            z += a;
        } else {
            // a bad key (negative, NaN, +inf) or one far above 2^m: the
            // exact update (it moves m to the key's exponent, or sets NaN)
            term_add<A, false>(m, u, z, k, v);
        }
    }
}

// term_add_lazy for the VEC pixels of a lane at once: the rare rescale is
// one branch for all of them (taken by a wave when any lane needs it), not
// one per pixel; the same arithmetic per pixel as term_add_lazy.
template <typename A, bool LOGW, int VEC>
__device__ __forceinline__ void terms_add_lazy(A (&m)[VEC], A (&u)[VEC], A (&z)[VEC],
                                               const A (&k)[VEC], const A (&v)[VEC]) {
    using M = NMath<A>;
    if constexpr (LOGW) {
        bool far = false;
#pragma unroll
        for (int i = 0; i < VEC; ++i) far |= k[i] - m[i] > A(kLazyLog);
        if (__builtin_expect(far, 0)) {
#pragma unroll
            for (int i = 0; i < VEC; ++i) {
                if (k[i] - m[i] > A(kLazyLog)) {
                    const A r = M::ex(m[i] - k[i]);
                    u[i] *= r;
                    z[i] *= r;
                    m[i] = k[i];
                }
            }
        }
#pragma unroll
        for (int i = 0; i < VEC; ++i) {
            const A a = M::ex(k[i] - m[i]);
            u[i] = fma_acc(a, v[i], u[i]);
            z[i] += a;
        }
    } else {
#pragma unroll
        for (int i = 0; i < VEC; ++i) term_add_lazy<A, false>(m[i], u[i], z[i], k[i], v[i]);
    }
}

// (m, u, z) := (m, u, z) merged with (m2, u2, z2).
template <typename A, bool LOGW>
__device__ __forceinline__ void state_merge(A& m, A& u, A& z, A m2, A u2, A z2) {
    using M = NMath<A>;
    if (LOGW) {
        const bool e1 = z == A(0), e2 = z2 == A(0);  // NaN (bad) is not empty
        const A mm = e1 ? m2 : (e2 ? m : (m > m2 ? m : m2));
        const A r1 = e1 ? A(0) : M::ex(m - mm);
        const A r2 = e2 ? A(0) : M::ex(m2 - mm);
        u = u * r1 + u2 * r2;
        z = z * r1 + z2 * r2;
        m = mm;
    } else {
        const int e1 = static_cast<int>(m), e2 = static_cast<int>(m2);
        const int mm = e1 > e2 ? e1 : e2;
        u = M::ldx(u, e1 - mm) + M::ldx(u2, e2 - mm);
        z = M::ldx(z, e1 - mm) + M::ldx(z2, e2 - mm);
        m = static_cast<A>(mm);
    }
}

template <typename A, bool LOGW>
__device__ __forceinline__ void state_final(A m, A u, A z, A& D, A& L) {
    if (z != z || (LOGW && m == Lim<A>::inf())) {  // bad key (NaN, or a +inf logit)
        D = Lim<A>::nan();
        L = Lim<A>::nan();
    } else if (z == A(0)) {
        D = A(0);
        L = -Lim<A>::inf();
    } else {
        D = u / z;
        // log C = m + log z, or (binary exponent m) m ln 2 + log z
        L = (LOGW ? m : m * A(0.693147180559945309)) + Lim<A>::lg(z);
    }
}

// Largest max(|dx|, |dy|) over the rows (only has_inverse rows when
// `only_inv`) that stay within the LDS halo; uniform across the workgroup.
template <int HALO = kRmax>
__device__ __forceinline__ int near_radius(const int4* shl, int S, bool only_inv) {
    const int lane = threadIdx.x & 63;
    int m = 0;
    for (int s = lane; s < S; s += 64) {
        const int4 r = shl[s];
        if (only_inv && r.z >= 0) continue;
        const int ax = r.x < 0 ? -r.x : r.x;
        const int ay = r.y < 0 ? -r.y : r.y;
        const int a = max(ax, ay);
        if (a <= HALO) m = max(m, a);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = max(m, __shfl_xor(m, o, 64));
    return __builtin_amdgcn_readfirstlane(m);
}

// Nontemporal weight loads: the fp64 forward 4-7% faster (c3 0.090 ->
// 0.085-0.087 ms), the fp32 backward on its 128-wide tiles 3% (c3 positive
// 0.642 -> 0.621 ms), the fp32 forward on 128-wide tiles 2% (on 64-wide
// tiles 13% slower: c3 0.326 -> 0.368 ms); the 16-bit forward 2% slower,
// the fp16 and fp64 backwards within the run-to-run spread (+-2%).  So:
// nontemporal in the fp64 forward and, with 32 lanes a row, in the fp32 forward
// and backward.  Those are the 128-wide tiles and the wide border's 64-wide
// ones of 2-pixel lanes, where it makes little difference (R = 10 1024^2 forward
// 331 us, plain 334, backward 452 and 456; R = 9 3 x 792^2 530 and 529, 893 and
// 860); the other 64-wide tiles load plainly.
template <typename T, int TPR>
constexpr bool kNormFwdNT = sizeof(T) == 8 || (sizeof(T) == 4 && TPR == 32);
template <typename T, int TPR>
constexpr bool kNormBwdNT = sizeof(T) == 4 && TPR == 32;
// The weight of pixel p for channel c from NH head planes: NH = 1 reads the
// plane as it is; NH > 1 forms sum_j mix[c][j] w_j[p] (the head-mixing
// product of the attention installers, applied where the weights are
// consumed, so no (S, B, C, H, W) stack is written and read).
template <typename T, int VEC, int NH, typename A>
__device__ __forceinline__ void mixed_pixels(PixSlot<T, VEC> (&slot)[NH], const A (&mixc)[NH],
                                             A (&wv)[VEC]) {
    slot_get_pixels<T, VEC>(slot[0], wv);
    if constexpr (NH > 1) {
#pragma unroll
        for (int k = 0; k < VEC; ++k) wv[k] *= mixc[0];
#pragma unroll
        for (int j = 1; j < NH; ++j) {
            A t[VEC];
            slot_get_pixels<T, VEC>(slot[j], t);
#pragma unroll
            for (int k = 0; k < VEC; ++k) wv[k] = fma_acc(mixc[j], t[k], wv[k]);
        }
    }
}

// Tile geometry with a HALO border: SGeo's, or rows at the plain LW pitch for
// the other borders where a row of lanes covers every bank at any pitch: the
// narrow one (fp64, 16 lanes of 8 bytes; the NSH_NARROW_HALO hint), so that
// three 256-lane workgroups share a CU, and the forward's wide one (32 lanes
// of 4 bytes; NSH_WIDE_HALO), whose four arrays would not fit otherwise.
template <int VEC, int ROWS, int TPR, int HALO, bool PLAIN = HALO != kRmax>
struct NTileGeo : SGeo<VEC, ROWS, TPR, true, HALO> {
    using Base = SGeo<VEC, ROWS, TPR, true, HALO>;
    static constexpr int PITCH = PLAIN ? Base::LW : Base::PITCH;
    static constexpr int TILE = Base::LH * PITCH;
};

// NH > 1: w is the head stack (S*B, NH, H, W), plane_step = B * NH * H * W,
// and mix the (C, NH) mixing matrix in the accumulator type.
template <typename T, int VEC, int TPR, int ROWS, int D, bool LOGW,
          int WPE = kScatterWavesPerEU<TPR * ROWS>, int NH = 1, int HALO = kRmax>
__global__ __launch_bounds__(TPR * ROWS, WPE) void
normalized_fwd_scatter_kernel(const T* __restrict__ x, const T* __restrict__ w,
                              const int64_t* __restrict__ shifts, int S, int codes, int C, int H,
                              int W, TileGrid tg, int64_t plane_step, acc_t<T>* __restrict__ Dout,
                              acc_t<T>* __restrict__ Lout, int* __restrict__ hdr,
                              acc_t<T>* __restrict__ spill, acc_t<T>* __restrict__ part,
                              int ring_stride, int64_t ntiles,
                              const acc_t<T>* __restrict__ mix, int* __restrict__ weights_ok) {
    using A = acc_t<T>;
    using G = NTileGeo<VEC, ROWS, TPR, HALO>;
    extern __shared__ __align__(16) unsigned char smem[];
    int4* shl = reinterpret_cast<int4*>(smem);
    A* xt = reinterpret_cast<A*>(smem + shift_lds_bytes(S));
    A* wm = xt + G::TILE;  // window of states (m, u, z)
    A* wu = wm + G::TILE;
    A* wz = wu + G::TILE;

    const int64_t t = xcd_tile(blockIdx.x, gridDim.x);
    const TileIdx ti = tile_of(t, tg, G::TH, G::TW, H, W);
    const int64_t HW = static_cast<int64_t>(H) * W;
    const int64_t off = ti.bc * HW;
    const T* xp = x + off;
    stage_shifts(shl, shifts, S, 3, H, W, codes);
    stage_tile<T, A>(xt, xp, H, W, ti.h0, ti.w0, G::LH, G::LW, G::PITCH, HALO);
    const int R = near_radius<HALO>(shl, S, true);
    if (blockIdx.x == 0 && threadIdx.x == 0) hdr[0] = R;  // for the fix-up
    const A m0 = empty_m<A, LOGW>();
    // the window is also used at R = 0 by a (0, 0) mirror row
    for (int i = threadIdx.x; i < G::TILE; i += blockDim.x) {
        wm[i] = m0;
        wu[i] = A(0);
        wz[i] = A(0);
    }
    __syncthreads();

    const int tx = threadIdx.x % TPR;
    const int ty = threadIdx.x / TPR;
    const int h = ti.h0 + ty;
    const LanePix<VEC, TPR> px = lane_pixels<VEC, TPR>(ti, ty, tx, W);
    const int lc = (ty + HALO) * G::PITCH + tx + HALO;  // pixel k at lc + k*TPR
    const int64_t b = ti.bc / C;
    const int64_t ch = ti.bc - b * C;
    const bool wsh = (codes & kCodesSharedW) != 0;
    // shift s adds s * wstep; head j of a mixed stack sits j planes further
    const T* w_bc = NH > 1 ? w + b * NH * HW : w + weight_plane(b, ch, C, wsh) * HW;
    const int64_t wstep = NH > 1 ? plane_step : weight_step(plane_step, C, wsh);
    A mixc[NH];
#pragma unroll
    for (int j = 0; j < NH; ++j) mixc[j] = NH > 1 ? mix[ch * NH + j] : A(1);

    A xo[VEC], sm[VEC], su[VEC], sz[VEC];
#pragma unroll
    for (int k = 0; k < VEC; ++k) {
        xo[k] = xt[lc + k * TPR];
        sm[k] = m0;
        su[k] = A(0);
        sz[k] = A(0);
    }
    // Weight prefetch ring (raw slots, promoted where consumed); the plane
    // of the next refill advances one plane per shift and the next shift's
    // record is read one shift ahead.
    PixSlot<T, VEC> wb[D][NH];
#pragma unroll
    for (int d = 0; d < D; ++d)
#pragma unroll
        for (int j = 0; j < NH; ++j)
            slot_load_pixels<T, VEC, TPR, kNormFwdNT<T, TPR>>(
                w_bc + j * HW + static_cast<int64_t>(min(d, S - 1)) * wstep, px, wb[d][j]);
    const T* wr = w_bc + static_cast<int64_t>(min(D, S - 1)) * wstep;
    ShiftRec rn = read_shift(shl, 0);

    // Interior tiles (every pixel inside the image and every q + s inside
    // it for all rows of the table) need no forward-box test and no mirror
    // mask: they run a select-free copy of the loop.
    const int R_all = table_radius(shl, S, false);
    const bool interior = ti.th == G::TH && ti.tw == G::TW && ti.h0 >= R_all && ti.h0 + G::TH + R_all <= H && ti.w0 >= R_all &&
                          ti.w0 + G::TW + R_all <= W;
    int last_dx = kClamp;
    // MODE 0: interior tile; 1: masks; 2: masks and forward-box rows
    auto step = [&](int s, PixSlot<T, VEC> (&slot)[NH], auto mode_tag) {
        constexpr int MODE = decltype(mode_tag)::value;
        const ShiftRec rc = rn;
        rn = read_shift(shl, min(s + 1, S - 1));
        A wv[VEC];
        mixed_pixels<T, VEC, NH, A>(slot, mixc, wv);
#pragma unroll
        for (int j = 0; j < NH; ++j)
            slot_load_pixels<T, VEC, TPR, kNormFwdNT<T, TPR>>(wr + j * HW, px, slot[j]);
        wr += s + D + 1 < S ? wstep : 0;
        if (shift_in_lds<HALO>(rc)) {
            const int op = lc + rc.dx * G::PITCH + rc.dy;  // window index of q + s
            if constexpr (MODE == 2) {
                // Forward box: a w_s[q] whose q + s leaves the image is a
                // masked key.  Only tiles this shift carries past the edge
                // test pixels.
                bool kept[VEC];
#pragma unroll
                for (int k = 0; k < VEC; ++k) kept[k] = true;
                if (rc.fbox && !tile_inside_n(ti.h0, ti.w0, G::TH, G::TW, H, W, rc.dx, rc.dy)) {
                    const bool frow = in_range(h + rc.dx, H);
#pragma unroll
                    for (int k = 0; k < VEC; ++k)
                        kept[k] = frow && in_range(ti.w0 + tx + k * TPR + rc.dy, W);
                }
#pragma unroll
                for (int k = 0; k < VEC; ++k) wv[k] = kept[k] ? wv[k] : masked_key<A, LOGW>();
            }
            {
                A xv[VEC];
#pragma unroll
                for (int k = 0; k < VEC; ++k) xv[k] = xt[op + k * TPR];
                terms_add_lazy<A, LOGW, VEC>(sm, su, sz, wv, xv);
            }
            if (rc.inv) {
                // Same dx: the wave's targets are its own rows shifted by dx,
                // disjoint from every other wave's; barrier only on a new dx.
                // Every lane merges (a masked key for a pixel outside the
                // image or a target outside the box changes nothing).  The
                // lane's VEC window states are read before any is written
                // (one LDS round trip per shift, not one per pixel).
                if (rc.dx != last_dx) {
                    lds_barrier();
                    last_dx = rc.dx;
                }
                const bool rok = rc.per || in_range(h + rc.dx, H);
                A m[VEC], u[VEC], z[VEC], kk[VEC], vv[VEC];
#pragma unroll
                for (int k = 0; k < VEC; ++k) {
                    const int i = op + k * TPR;
                    m[k] = wm[i];
                    u[k] = wu[i];
                    z[k] = wz[i];
                    if constexpr (MODE == 0) {
                        kk[k] = wv[k];
                        vv[k] = xo[k];
                    } else {
                        const bool ok = px.act[k] && rok &&
                                        (rc.per || in_range(ti.w0 + tx + k * TPR + rc.dy, W));
                        kk[k] = ok ? wv[k] : masked_key<A, LOGW>();
                        vv[k] = ok ? xo[k] : A(0);
                    }
                }
                terms_add_lazy<A, LOGW, VEC>(m, u, z, kk, vv);
#pragma unroll
                for (int k = 0; k < VEC; ++k) {
                    const int i = op + k * TPR;
                    wm[i] = m[k];
                    wu[i] = u[k];
                    wz[i] = z[k];
                }
            }
        }
    };
    auto ring = [&](auto mode_tag) {
        const int S_ring = S - S % D;
        for (int s0 = 0; s0 < S_ring; s0 += D) {
#pragma unroll
            for (int d = 0; d < D; ++d) step(s0 + d, wb[d], mode_tag);
        }
#pragma unroll
        for (int d = 0; d < D; ++d)
            if (S_ring + d < S) step(S_ring + d, wb[d], mode_tag);
    };
    if (interior)
        ring(std::integral_constant<int, 0>{});
    else if (table_any_fbox(shl, S))
        ring(std::integral_constant<int, 2>{});
    else
        ring(std::integral_constant<int, 1>{});
    // Shifts beyond the halo: gather form (forward x and mirror terms read
    // from HBM), kept out of the ring loop.
    auto weight_at = [&](const T* wp, uint32_t i) {
        A v = to_acc(wp[i]);
        if constexpr (NH > 1) {
            v *= mixc[0];
#pragma unroll
            for (int j = 1; j < NH; ++j) v = fma_acc(mixc[j], to_acc(wp[j * HW + i]), v);
        }
        return v;
    };
    for (int s = 0; s < S && px.any; ++s) {
        const ShiftRec rc = read_shift(shl, s);
        if (shift_in_lds<HALO>(rc)) continue;
        const T* wp = w_bc + static_cast<int64_t>(s) * wstep;
        int hp = h + rc.dxm;
        hp -= hp >= H ? H : 0;
        int hm = h - rc.dxm;
        hm += hm < 0 ? H : 0;
        const bool irow = rc.per || in_range(h - rc.dx, H);
#pragma unroll
        for (int k = 0; k < VEC; ++k) {
            if (!px.act[k]) continue;
            const int wq = ti.w0 + tx + k * TPR;
            int wj = wq + rc.dym;
            wj -= wj >= W ? W : 0;
            const A wq_ = weight_at(wp, px.own[k]);
            term_add<A, LOGW>(sm[k], su[k], sz[k],
                              fwd_kept(rc, h, wq, H, W) ? wq_ : masked_key<A, LOGW>(),
                              to_acc(xp[static_cast<uint32_t>(hp) * W + wj]));
            if (rc.inv && irow && (rc.per || in_range(wq - rc.dy, W))) {
                int wm_ = wq - rc.dym;
                wm_ += wm_ < 0 ? W : 0;
                const uint32_t src = static_cast<uint32_t>(hm) * W + wm_;
                term_add<A, LOGW>(sm[k], su[k], sz[k], weight_at(wp, src), to_acc(xp[src]));
            }
        }
    }

    // the head-mixing kernels (NH > 1) are never asked (weights_ok is null), and
    // their registers are full: with the check in them four heads spilled 22 to
    // 27 registers a lane
    if (NH == 1 && weights_ok != nullptr) {
        // every weight the box kept went into its own pixel's state
        bool bad = false;
#pragma unroll
        for (int k = 0; k < VEC; ++k)
            bad |= px.act[k] && (sz[k] != sz[k] || (LOGW && sm[k] == Lim<A>::inf()));
        // The ones it dropped are read again here, a batch of shifts in
        // flight (a pixel that keeps its weight re-reads its plane's first
        // element): tested in the ring loop they made every forward with the
        // box 5% (fp16 logits) to 19% (rows beyond the border) slower.
        if (!interior && table_any_fbox(shl, S)) {
            constexpr int NB = 8;
            for (int s0 = 0; s0 < S; s0 += NB) {
                A v[NB][VEC];
#pragma unroll
                for (int i = 0; i < NB; ++i) {
                    const ShiftRec rc = read_shift(shl, min(s0 + i, S - 1));
                    const T* wp = w_bc + static_cast<int64_t>(min(s0 + i, S - 1)) * wstep;
#pragma unroll
                    for (int k = 0; k < VEC; ++k) {
                        const bool kept = fwd_kept(rc, h, ti.w0 + tx + k * TPR, H, W);
                        v[i][k] = to_acc(*elem_ptr(wp, kept ? 0u : px.own[k]));
                    }
                }
#pragma unroll
                for (int i = 0; i < NB; ++i)
#pragma unroll
                    for (int k = 0; k < VEC; ++k) bad |= key_bad<A, LOGW>(v[i][k]);
            }
        }
        if (bad) *weights_ok = 0;
    }
    __syncthreads();
    const int th = ti.th, tw = ti.tw;
    A* pm = part + 3 * t * ring_stride;
#pragma unroll
    for (int k = 0; k < VEC; ++k) {
        if (!px.act[k]) continue;
        const int i = lc + k * TPR;
        state_merge<A, LOGW>(sm[k], su[k], sz[k], wm[i], wu[i], wz[i]);
        if (R > 0) {
            const int slot = ring_slot(ty, tx + k * TPR, th, tw, R);
            if (slot >= 0) {  // finished by the fix-up
                pm[slot] = sm[k];
                pm[ring_stride + slot] = su[k];
                pm[2 * ring_stride + slot] = sz[k];
                continue;
            }
        }
        A Dv, Lv;
        state_final<A, LOGW>(sm[k], su[k], sz[k], Dv, Lv);
        Dout[off + px.own[k]] = Dv;
        Lout[off + px.own[k]] = Lv;
    }
    if (R == 0) return;
    const int n = spill_count(th, tw, R);
    A* s0p = spill + t * G::SPILL;
    A* s1p = spill + (ntiles + t) * G::SPILL;
    A* s2p = spill + (2 * ntiles + t) * G::SPILL;
    for (int e = threadIdx.x; e < n; e += blockDim.x) {
        int i, j;
        spill_coords(e, th, tw, R, i, j);
        const int li = (i + HALO) * G::PITCH + j + HALO;
        s0p[e] = wm[li];
        s1p[e] = wu[li];
        s2p[e] = wz[li];
    }
}

// Finishes the ring pixels of the forward: own partial state merged with
// the neighbouring tiles' spilled window states (fixed order), then D and
// log_C.
template <typename A, bool LOGW>
__global__ __launch_bounds__(256) void normalized_fixup_kernel(
    int H, int W, int TH, int TW, TileGrid tg, int spill_stride, int ring_stride,
    const int* __restrict__ hdr, const A* __restrict__ spill, const A* __restrict__ part,
    int64_t ntiles, A* __restrict__ Dout, A* __restrict__ Lout) {
    const int R = __builtin_amdgcn_readfirstlane(hdr[0]);
    if (R == 0) return;
    const FixTile f = fix_tile(blockIdx.x, H, W, TH, TW, tg);
    const int64_t HW = static_cast<int64_t>(H) * W;
    const A* pm = part + 3 * static_cast<int64_t>(blockIdx.x) * ring_stride;
    int lg;
    if (fix_slots_ok(f, R, TW, false, lg)) {
        // ring tiles: the slot enumeration, kFixBatch slots per lane with
        // all their loads issued before any merge
        const FixRing g = fix_ring<false>(f, R, lg, HW, W, spill_stride);
        const int64_t qstride = ntiles * spill_stride;
        const int step = static_cast<int>(blockDim.x);
        for (int s0 = threadIdx.x; s0 < g.n; s0 += step * kFixBatch) {
            int lr[kFixBatch], lc[kFixBatch];
            bool act[kFixBatch];
            uint32_t pp[kFixBatch];
            int64_t e[kFixBatch][3];
            A st[kFixBatch][3], sv[kFixBatch][3][3];
#pragma unroll
            for (int k = 0; k < kFixBatch; ++k) {
                fix_slot<false>(f, g, s0 + k * step, W, lr[k], lc[k], act[k], pp[k], e[k]);
                const int ri = ring_slot(lr[k], lc[k], f.th, f.tw, R);
#pragma unroll
                for (int q = 0; q < 3; ++q) {
                    st[k][q] = pm[q * ring_stride + ri];
#pragma unroll
                    for (int c = 0; c < 3; ++c)
                        sv[k][q][c] = spill[e[k][c] >= 0 ? q * qstride + e[k][c] : 0];
                }
            }
#pragma unroll
            for (int k = 0; k < kFixBatch; ++k) {
                if (!act[k]) continue;
                A m = st[k][0], u = st[k][1], z = st[k][2];
#pragma unroll
                for (int c = 0; c < 3; ++c)
                    if (e[k][c] >= 0)
                        state_merge<A, LOGW>(m, u, z, sv[k][0][c], sv[k][1][c], sv[k][2][c]);
                A Dv, Lv;
                state_final<A, LOGW>(m, u, z, Dv, Lv);
                Dout[g.pb + pp[k]] = Dv;
                Lout[g.pb + pp[k]] = Lv;
            }
        }
        return;
    }
    const int n = ring_count(f.th, f.tw, R);
    for (int idx = threadIdx.x; idx < n; idx += blockDim.x) {
        int lr, lc;
        ring_pixel(idx, f.th, f.tw, R, lr, lc);
        A m = pm[idx], u = pm[ring_stride + idx], z = pm[2 * ring_stride + idx];
        spill_visit(f, R, lr, lc, [&](int64_t tn, int e) {
            state_merge<A, LOGW>(m, u, z, spill[tn * spill_stride + e],
                                 spill[(ntiles + tn) * spill_stride + e],
                                 spill[(2 * ntiles + tn) * spill_stride + e]);
        });
        A Dv, Lv;
        state_final<A, LOGW>(m, u, z, Dv, Lv);
        const int64_t p = f.bc * HW + static_cast<int64_t>(f.h0 + lr) * W + (f.w0 + lc);
        Dout[p] = Dv;
        Lout[p] = Lv;
    }
}

// Backward.  LDS: x; L (log weights) or E = exp(-L) (positive weights);
// alpha = gD; beta = gLogC - gD D (so score(o, v) = alpha[o] v + beta[o]);
// and the x-gradient window.  With a 16-bit T the gx partial sums go to
// `gxp` (accumulator type) and the fix-up rounds once.
template <typename A, bool LOGW>
__device__ __forceinline__ A frac_tile(A w, A l) {
    // f(w, L): log weights exp(w - L); positive weights w E with l = E = exp(-L)
    if (LOGW) return (w == -Lim<A>::inf() || l == -Lim<A>::inf()) ? A(0) : Lim<A>::ex(w - l);
    return (w == A(0) || l == Lim<A>::inf()) ? A(0) : w * l;
}

// Log keys of the backward's fractions f = exp(l - L): the staged L is
// log_key(L) = L log2(e) (fp32; fp64 keeps natural units), with an empty
// row's L = -inf staged as +inf, and a term's logit enters as
// log_scale(l) = l log2(e); then f = exp2(log_scale(l) - log_key(L)) is 0
// for an empty row without a test (exp2(-inf)), and a masked logit (-inf) is
// tested once by the caller.  One multiply per term serves both fractions
// of a term (own and mirror output).
template <typename A>
__device__ __forceinline__ A log_scale(A l) {
    if constexpr (sizeof(A) == 4) return l * 1.44269504088896341f;
    return l;
}
template <typename A>
__device__ __forceinline__ A log_key(A L) {
    return L == -Lim<A>::inf() ? Lim<A>::inf() : log_scale<A>(L);
}
template <typename A>
__device__ __forceinline__ A frac_log(A kw, A key) {
    if constexpr (sizeof(A) == 4) return __builtin_amdgcn_exp2f(kw - key);
    return Lim<A>::ex(kw - key);
}

// CONTIG (W a multiple of VEC = 4, or 2 on the wide border, and tensors aligned
// for it): lane tx owns VEC consecutive pixels of its row, moved with one
// vector load or store per shift, and the LDS tiles use the de-interleaved
// columns of BwdLayout (conflict-free for these lanes).  Otherwise the lanes
// are strided (pixels tx, tx + TPR, ...) with row-major tiles.
// NTS: streaming stores of gw, where whole rows are whole 128-byte lines or the
// lanes store fp32 vectors, as in accumulate_uz's backward (R = 5, streaming ->
// plain elsewhere: 3 x 1100 x 1500 fp16 551 -> 443 us, 8 x 3 x 250^2 fp32 267 ->
// 237 us, 1500^2 fp64 687 -> 583 us; kept streaming: 1500^2 fp32 315 against 336).
template <typename T, int VEC, int TPR, int ROWS, int D, bool LOGW, bool CONTIG, bool NTS,
          int WPE = kScatterWavesPerEU<TPR * ROWS>, int HALO = kRmax>
__global__ __launch_bounds__(TPR * ROWS, WPE) void
normalized_bwd_scatter_kernel(const T* __restrict__ x, const T* __restrict__ w,
                              const acc_t<T>* __restrict__ Dg, const acc_t<T>* __restrict__ Lg,
                              const acc_t<T>* __restrict__ gDg, const acc_t<T>* __restrict__ gLg,
                              const int64_t* __restrict__ shifts, int S, int codes, int C, int H,
                              int W, TileGrid tg, int64_t plane_step, T* __restrict__ gx,
                              acc_t<T>* __restrict__ gxp, T* __restrict__ gw,
                              int* __restrict__ hdr, acc_t<T>* __restrict__ spill) {
    using A = acc_t<T>;
    using G = NTileGeo<VEC, ROWS, TPR, HALO, (HALO < kRmax)>;
    static_assert(HALO >= kRmax || !CONTIG, "the narrow border is built for strided lanes");
    static_assert(!CONTIG || VEC == 4 || VEC == 2, "the contiguous form moves vectors");
    // Column offset within a row: de-interleaved for the contiguous lanes
    // (the strided SGeo pitch is the BwdLayout pitch), row-major otherwise.
    using L = BwdLayout<VEC, G::LW, G::PITCH>;
    auto colm = [](int j) { return CONTIG ? L::col(j) : j; };
    static_assert(!CONTIG || L::PITCH == G::PITCH, "de-interleaved rows use the strided pitch");
    extern __shared__ __align__(16) unsigned char smem[];
    int4* shl = reinterpret_cast<int4*>(smem);
    A* xt = reinterpret_cast<A*>(smem + shift_lds_bytes(S));
    A* lt = xt + G::TILE;
    A* at = lt + G::TILE;
    A* bt = at + G::TILE;
    A* mg = bt + G::TILE;

    const int64_t t = xcd_tile(blockIdx.x, gridDim.x);
    const TileIdx ti = tile_of(t, tg, G::TH, G::TW, H, W);
    const int64_t HW = static_cast<int64_t>(H) * W;
    const int64_t off = ti.bc * HW;
    const T* xp = x + off;
    const A* Dp = Dg + off;
    const A* Lp = Lg + off;
    const A* gDp = gDg + off;
    const A* gLp = gLg + off;
    stage_shifts(shl, shifts, S, 3, H, W, codes);
    {
        const bool cheap = H >= G::LH && W >= G::LW;
        for (int i = threadIdx.x; i < G::LH * G::LW; i += blockDim.x) {
            const int r = i / G::LW;
            const int cc = i - r * G::LW;
            int gh = ti.h0 - HALO + r;
            int gw_ = ti.w0 - HALO + cc;
            if (cheap) {
                gh = wrap1(gh, H);
                gw_ = wrap1(gw_, W);
            } else {
                gh = static_cast<int>(mod_pos(gh, H));
                gw_ = static_cast<int>(mod_pos(gw_, W));
            }
            const uint32_t g = static_cast<uint32_t>(gh) * static_cast<uint32_t>(W) +
                               static_cast<uint32_t>(gw_);
            const int li = r * G::PITCH + colm(cc);
            const A gd = gDp[g];
            xt[li] = to_acc(xp[g]);
            lt[li] = LOGW ? log_key<A>(Lp[g]) : Lim<A>::ex(-Lp[g]);
            at[li] = gd;
            bt[li] = gLp[g] - gd * Dp[g];
        }
    }
    const int R = near_radius<HALO>(shl, S, false);
    if (blockIdx.x == 0 && threadIdx.x == 0) hdr[0] = R;  // for the fix-up
    lds_zero(mg, G::TILE);
    __syncthreads();

    const int tx = threadIdx.x % TPR;
    const int ty = threadIdx.x / TPR;
    const int h = ti.h0 + ty;
    // The lane's pixels: column, activity and in-plane offset of pixel k,
    // and its LDS index displaced by (dx, dy).
    const LanePix<VEC, TPR> px = lane_pixels<VEC, TPR>(ti, ty, tx, W);  // strided form
    const int wq0 = ti.w0 + tx * VEC;                                          // contiguous form
    const bool cact = ty < ti.th && tx * VEC < ti.tw;
    const uint32_t cown = static_cast<uint32_t>(cact ? h : 0) * static_cast<uint32_t>(W) +
                          static_cast<uint32_t>(cact ? wq0 : 0);
    auto pcol = [&](int k) { return CONTIG ? wq0 + k : ti.w0 + tx + k * TPR; };
    auto pact = [&](int k) { return CONTIG ? cact : px.act[k]; };
    auto pown = [&](int k) { return CONTIG ? cown + k : px.own[k]; };
    const int lrow = (ty + HALO) * G::PITCH + (CONTIG ? tx : 0);
    auto lidx = [&](int k, int dx, int dy) {
        return lrow + dx * G::PITCH + (CONTIG ? colm(HALO + k + dy) : tx + HALO + k * TPR + dy);
    };
    const int64_t b = ti.bc / C;
    const bool wsh = (codes & kCodesSharedW) != 0;
    const T* w_bc = w + weight_plane(b, ti.bc - b * C, C, wsh) * HW;
    const int64_t wstep = weight_step(plane_step, C, wsh);
    T* g_bc = gw + ti.bc * HW;  // the gradient has every channel
    // Weight prefetch ring: raw slots (promoted where consumed), one vector
    // per lane (contiguous) or one element per pixel (strided).
    using Slot = std::conditional_t<CONTIG, SlotRaw<T, VEC>, PixSlot<T, VEC>>;
    auto slot_fill = [&](const T* wp, Slot& sl) {
        if constexpr (CONTIG)
            slot_load_at<T, VEC, kNormBwdNT<T, TPR>>(wp, cown * static_cast<uint32_t>(sizeof(T)),
                                                       sl);
        else
            slot_load_pixels<T, VEC, TPR, kNormBwdNT<T, TPR>>(wp, px, sl);
    };
    auto slot_take = [&](const Slot& sl, A (&wv)[VEC]) {
        if constexpr (CONTIG)
            slot_get<T, VEC>(sl, wv);
        else
            slot_get_pixels<T, VEC>(sl, wv);
    };

    A xo[VEC], lo[VEC], ao[VEC], bo[VEC], gxa[VEC];
#pragma unroll
    for (int k = 0; k < VEC; ++k) {
        const int i = lidx(k, 0, 0);
        xo[k] = xt[i];
        lo[k] = lt[i];
        ao[k] = at[i];
        bo[k] = bt[i];
        gxa[k] = A(0);
    }
    Slot wb[D];
#pragma unroll
    for (int d = 0; d < D; ++d) slot_fill(w_bc + static_cast<int64_t>(min(d, S - 1)) * wstep, wb[d]);
    // the next refill's plane and the next shift's record, advanced per
    // shift; the gw plane of the current shift
    const T* wr = w_bc + static_cast<int64_t>(min(D, S - 1)) * wstep;
    ShiftRec rn = read_shift(shl, 0);
    T* gs = g_bc;

    // gw_s[q] for one pixel given the neighbour values at q + s.  Log
    // weights: the staged L are log keys (log_key), so both fractions are
    // exp of one difference of the scaled logit (frac_log), with a single
    // test of the mask.
    auto grad_w = [&](int k, A wv, A xf, A lp, A ap, A bp, bool okp, A& fo) -> A {
        const bool masked = LOGW ? wv == -Lim<A>::inf() : wv == A(0);
        A Ff, Fi;
        if constexpr (LOGW) {
            const A kw = log_scale<A>(wv);
            fo = masked ? A(0) : frac_log<A>(kw, lo[k]);  // f(w_s[q], L[q])
            Ff = fo;
            Fi = masked ? A(0) : frac_log<A>(kw, lp);     // f(w_s[q], L[q+s])
        } else {
            fo = frac_tile<A, LOGW>(wv, lo[k]);  // f(w_s[q], L[q])
            Ff = lo[k];                          // F(L[q])
            Fi = lp;
        }
        const A sf = fma_acc(ao[k], xf, bo[k]);   // score(q, x[q+s])
        const A si = fma_acc(ap, xo[k], bp);      // score(q+s, x[q])
        const A gv = fma_acc(Ff, sf, okp ? Fi * si : A(0));
        if (okp) gxa[k] = fma_acc(LOGW ? Fi : frac_tile<A, LOGW>(wv, lp), ap, gxa[k]);
        return masked ? A(0) : gv;
    };

    // Interior tiles (every pixel and every q + s inside the image for all
    // rows of the table): no forward-box test and no mirror mask.
    const int R_all = table_radius(shl, S, false);
    const bool interior = ti.th == G::TH && ti.tw == G::TW && ti.h0 >= R_all && ti.h0 + G::TH + R_all <= H && ti.w0 >= R_all &&
                          ti.w0 + G::TW + R_all <= W;
    int last_dx = kClamp;
    auto step = [&](int s, Slot& slot, auto fast_tag) {
        constexpr bool FAST = decltype(fast_tag)::value;
        const ShiftRec rc = rn;
        rn = read_shift(shl, min(s + 1, S - 1));
        A wv[VEC];
        slot_take(slot, wv);
        slot_fill(wr, slot);
        wr += s + D + 1 < S ? wstep : 0;
        if (shift_in_lds<HALO>(rc)) {
            if (rc.dx != last_dx) {
                lds_barrier();
                last_dx = rc.dx;
            }
            const bool rok = rc.inv && (rc.per || in_range(h + rc.dx, H));
            A gv[VEC];
#pragma unroll
            for (int k = 0; k < VEC; ++k) {
                const int i = lidx(k, rc.dx, rc.dy);
                A fo;
                if constexpr (FAST) {
                    gv[k] = grad_w(k, wv[k], xt[i], lt[i], at[i], bt[i], rc.inv, fo);
                    if constexpr (!CONTIG)
                        store_elem_at<T, NTS>(gs, px.own[k] * static_cast<uint32_t>(sizeof(T)),
                                               from_acc<T>(gv[k]));
                    mg[i] += fo * ao[k];
                } else {
                    const bool okp = rok && (rc.per || in_range(pcol(k) + rc.dy, W));
                    const A wk = fwd_kept(rc, h, pcol(k), H, W) ? wv[k] : masked_key<A, LOGW>();
                    gv[k] = grad_w(k, wk, xt[i], lt[i], at[i], bt[i], okp, fo);
                    if constexpr (!CONTIG)
                        if (px.act[k])
                            store_elem_at<T, NTS>(
                                gs, px.own[k] * static_cast<uint32_t>(sizeof(T)), from_acc<T>(gv[k]));
                    // x-gradient term of q + s: f(w_s[q], L[q]) gD[q]
                    mg[i] += pact(k) ? fo * ao[k] : A(0);
                }
            }
            if constexpr (CONTIG)
                if (FAST || cact)
                    store_acc_at<T, VEC, NTS>(gs, cown * static_cast<uint32_t>(sizeof(T)), gv);
        }
        gs += plane_step;
    };
    auto ring = [&](auto fast_tag) {
        const int S_ring = S - S % D;
        for (int s0 = 0; s0 < S_ring; s0 += D) {
#pragma unroll
            for (int d = 0; d < D; ++d) step(s0 + d, wb[d], fast_tag);
        }
#pragma unroll
        for (int d = 0; d < D; ++d)
            if (S_ring + d < S) step(S_ring + d, wb[d], fast_tag);
    };
    if (interior)
        ring(std::true_type{});
    else
        ring(std::false_type{});
    // Shifts beyond the halo: gather form, neighbour values from HBM.
    for (int s = 0; s < S && (CONTIG ? cact : px.any); ++s) {
        const ShiftRec rc = read_shift(shl, s);
        if (shift_in_lds<HALO>(rc)) continue;
        const T* wp = w_bc + static_cast<int64_t>(s) * wstep;
        T* gs = g_bc + static_cast<int64_t>(s) * plane_step;
        int hp = h + rc.dxm;
        hp -= hp >= H ? H : 0;
        int hm = h - rc.dxm;
        hm += hm < 0 ? H : 0;
        const bool rok = rc.inv && (rc.per || in_range(h + rc.dx, H));
#pragma unroll
        for (int k = 0; k < VEC; ++k) {
            if (!pact(k)) continue;
            const int wq = pcol(k);
            int wj = wq + rc.dym;
            wj -= wj >= W ? W : 0;
            int wm = wq - rc.dym;
            wm += wm < 0 ? W : 0;
            const uint32_t ip = static_cast<uint32_t>(hp) * W + wj;
            const uint32_t im = static_cast<uint32_t>(hm) * W + wm;
            const bool okp = rok && (rc.per || in_range(wq + rc.dy, W));
            const A lp = LOGW ? log_key<A>(Lp[ip]) : Lim<A>::ex(-Lp[ip]);
            const A gdp = gDp[ip];
            A fo;
            const A wk = fwd_kept(rc, h, wq, H, W) ? to_acc(*elem_ptr(wp, pown(k)))
                                                   : masked_key<A, LOGW>();
            const A g = grad_w(k, wk, to_acc(xp[ip]), lp, gdp, gLp[ip] - gdp * Dp[ip], okp, fo);
            store_elem_nt<T>(elem_ptr(gs, pown(k)), from_acc<T>(g));
            // x-gradient term from o = (q - s) mod: f(w_s[o], L[o]) gD[o]
            const A lm = LOGW ? Lp[im] : Lim<A>::ex(-Lp[im]);
            const A wo = fwd_kept_src(rc, h, wq, H, W) ? to_acc(wp[im]) : masked_key<A, LOGW>();
            gxa[k] = fma_acc(frac_tile<A, LOGW>(wo, lm), gDp[im], gxa[k]);
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < VEC; ++k) {
        if (!pact(k)) continue;
        const A v = gxa[k] + mg[lidx(k, 0, 0)];
        if (gxp != nullptr)
            gxp[off + pown(k)] = v;
        else
            gx[off + pown(k)] = from_acc<T>(v);
    }
    if (R == 0) return;
    const int th = ti.th, tw = ti.tw;
    const int n = spill_count(th, tw, R);
    A* sg = spill + t * G::SPILL;
    for (int e = threadIdx.x; e < n; e += blockDim.x) {
        int i, j;
        spill_coords(e, th, tw, R, i, j);
        sg[e] = mg[(i + HALO) * G::PITCH + colm(j + HALO)];
    }
}

// Backward of channel-shared weights, the weights' own gradient (the sum over
// the channels) formed here.  The per-channel kernel above runs one workgroup
// per channel: each reads the weights and forms the fractions f(w, L) again
// (the degree of shared weights is the same for every channel, so L is read
// from channel 0), writes a gradient plane of its own, and the C planes per
// shift are read back and summed.  Here a workgroup takes the NC channels of
// its tile: one key array, and x, alpha, beta and the gx window per channel,
// 4 NC + 1 LDS arrays, on 64 x 16 tiles of 1024 lanes, one pixel each (133 KB
// at NC = 3; four channels would not fit).  Per channel with the sum, and
// here: 8 x 3 x 250^2 R = 5 fp32 330 and 112 us (3.1 TB/s of weights and their
// gradient), fp16 207 and 104; 1024^2 C = 3 R = 6 fp32 690 and 283; 2 channels
// of 321 x 481 R = 6 256 and 113.  Rows beyond the border take the gather form
// here too, and that is still the faster side of the two for tables that the
// per-channel kernels serve on the 16-pixel border (R = 10, 221 rows, fp32:
// 1230 and 494 us; 69 rows of radius 16 under NSH_WIDE_HALO, which the Python
// layer does not set for so few, 832 and 215).  Bound by the loop's
// LDS accesses (13 reads and 3 writes per pixel and row) at 16 waves per CU:
// fp16 takes 0.93 of fp32's time.
// beta stays per channel, so that each score is formed as above: with the
// channels' beta summed at the load the scores' error against 64 bits grew by
// 4% (x of mean 5, C = 3) to 22% (maximum, C = 4).
constexpr int kNShRows = 16, kNShTpr = 64, kNShDepth = 4;

template <typename T, int NC, bool LOGW>
__global__ __launch_bounds__(kNShTpr * kNShRows, 4) void normalized_bwd_shared_kernel(
    const T* __restrict__ x, const T* __restrict__ w, const acc_t<T>* __restrict__ Dg,
    const acc_t<T>* __restrict__ Lg, const acc_t<T>* __restrict__ gDg,
    const acc_t<T>* __restrict__ gLg, const int64_t* __restrict__ shifts, int S, int codes, int H,
    int W, TileGrid tg, int64_t wstep, T* __restrict__ gx, acc_t<T>* __restrict__ gxp,
    T* __restrict__ gw, int* __restrict__ hdr, acc_t<T>* __restrict__ spill) {
    using A = acc_t<T>;
    using G = SGeo<1, kNShRows, kNShTpr>;
    constexpr int D = kNShDepth, HALO = kRmax;
    extern __shared__ __align__(16) unsigned char smem[];
    int4* shl = reinterpret_cast<int4*>(smem);
    A* lt = reinterpret_cast<A*>(smem + shift_lds_bytes(S));  // L key or E
    A* xt = lt + G::TILE;                                      // NC tiles each
    A* at = xt + NC * G::TILE;
    A* bt = at + NC * G::TILE;
    A* mg = bt + NC * G::TILE;

    const int64_t t = xcd_tile(blockIdx.x, gridDim.x);
    const TileIdx ti = tile_of(t, tg, G::TH, G::TW, H, W);  // ti.bc: the batch entry
    const int64_t HW = static_cast<int64_t>(H) * W;
    const int64_t off = ti.bc * NC * HW;  // channel 0 of this batch entry
    stage_shifts(shl, shifts, S, 3, H, W, codes);
    {
        const bool cheap = H >= G::LH && W >= G::LW;
        for (int i = threadIdx.x; i < G::LH * G::LW; i += blockDim.x) {
            const int64_t g = off + halo_offset(i, G::LW, ti.h0, ti.w0, H, W, cheap);
            const int r = i / G::LW;
            const int li = r * G::PITCH + (i - r * G::LW);
            A d[NC], gd[NC], gl[NC];
            T xv[NC];
            const A L = Lg[g];
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                xv[c] = x[g + c * HW];
                gd[c] = gDg[g + c * HW];
                gl[c] = gLg[g + c * HW];
                d[c] = Dg[g + c * HW];
            }
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                xt[c * G::TILE + li] = to_acc(xv[c]);
                at[c * G::TILE + li] = gd[c];
                bt[c * G::TILE + li] = gl[c] - gd[c] * d[c];
            }
            lt[li] = LOGW ? log_key<A>(L) : Lim<A>::ex(-L);
        }
    }
    const int R = near_radius(shl, S, false);
    if (blockIdx.x == 0 && threadIdx.x == 0) hdr[0] = R;  // for the fix-up
    lds_zero(mg, NC * G::TILE);
    __syncthreads();

    const int tx = threadIdx.x % kNShTpr;
    const int ty = threadIdx.x / kNShTpr;
    const int h = ti.h0 + ty, wq = ti.w0 + tx;
    const bool act = ty < ti.th && tx < ti.tw;
    const uint32_t own = act ? static_cast<uint32_t>(h) * static_cast<uint32_t>(W) + wq : 0u;
    const uint32_t own_b = own * static_cast<uint32_t>(sizeof(T));
    const int li = (ty + HALO) * G::PITCH + tx + HALO;
    const T* w_b = w + ti.bc * HW;
    T* g_b = gw + ti.bc * HW;

    A xo[NC], ao[NC], bo[NC], gxa[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        xo[c] = xt[c * G::TILE + li];
        ao[c] = at[c * G::TILE + li];
        bo[c] = bt[c * G::TILE + li];
        gxa[c] = A(0);
    }
    const A lo = lt[li];
    SlotRaw<T, 1> wb[D];  // weight prefetch ring, as in the kernels above
#pragma unroll
    for (int d = 0; d < D; ++d)
        slot_load_at<T, 1>(w_b + static_cast<int64_t>(min(d, S - 1)) * wstep, own_b, wb[d]);
    const T* wr = w_b + static_cast<int64_t>(min(D, S - 1)) * wstep;
    ShiftRec rn = read_shift(shl, 0);
    T* gs = g_b;

    // The terms of one weight: its gradient, summed over the channels, from
    // the neighbour's values; the mirror's x gradient; fo = f(w, L[q]).
    auto terms = [&](A wv, const A (&xf)[NC], A lp, const A (&ap)[NC], const A (&bp)[NC],
                     bool okp, A& fo) -> A {
        const bool masked = LOGW ? wv == -Lim<A>::inf() : wv == A(0);
        A Ff, Fi, fi;
        if constexpr (LOGW) {
            const A kw = log_scale<A>(wv);
            fo = masked ? A(0) : frac_log<A>(kw, lo);
            fi = masked ? A(0) : frac_log<A>(kw, lp);
            Ff = fo;
            Fi = fi;
        } else {
            fo = frac_tile<A, false>(wv, lo);
            fi = frac_tile<A, false>(wv, lp);
            Ff = lo;
            Fi = lp;
        }
        A sf = A(0), si = A(0);
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            sf += fma_acc(ao[c], xf[c], bo[c]);
            si += fma_acc(ap[c], xo[c], bp[c]);
            if (okp) gxa[c] = fma_acc(fi, ap[c], gxa[c]);
        }
        const A gv = fma_acc(Ff, sf, okp ? Fi * si : A(0));
        return masked ? A(0) : gv;
    };
    const int R_all = table_radius(shl, S, false);
    const bool interior = ti.th == G::TH && ti.tw == G::TW && ti.h0 >= R_all &&
                          ti.h0 + G::TH + R_all <= H && ti.w0 >= R_all &&
                          ti.w0 + G::TW + R_all <= W;
    int last_dx = kClamp;
    auto step = [&](int s, SlotRaw<T, 1>& slot, auto fast_tag) {
        constexpr bool FAST = decltype(fast_tag)::value;
        const ShiftRec rc = rn;
        rn = read_shift(shl, min(s + 1, S - 1));
        A w1[1];
        slot_get<T, 1>(slot, w1);
        slot_load_at<T, 1>(wr, own_b, slot);
        wr += s + D + 1 < S ? wstep : 0;
        if (shift_in_lds(rc)) {
            if (rc.dx != last_dx) {
                lds_barrier();
                last_dx = rc.dx;
            }
            const int i = li + rc.dx * G::PITCH + rc.dy;
            const bool okp = rc.inv && (FAST || rc.per ||
                                        (in_range(h + rc.dx, H) && in_range(wq + rc.dy, W)));
            const A wv = FAST || fwd_kept(rc, h, wq, H, W) ? w1[0] : masked_key<A, LOGW>();
            A xf[NC], ap[NC], bp[NC], m[NC], fo;
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                xf[c] = xt[c * G::TILE + i];
                ap[c] = at[c * G::TILE + i];
                bp[c] = bt[c * G::TILE + i];
                m[c] = mg[c * G::TILE + i];
            }
            const A g = terms(wv, xf, lt[i], ap, bp, okp, fo);
            if (FAST || act) store_elem_at<T, false>(gs, own_b, from_acc<T>(g));
#pragma unroll
            for (int c = 0; c < NC; ++c)
                mg[c * G::TILE + i] = m[c] + (FAST || act ? fo * ao[c] : A(0));
        }
        gs += wstep;
    };
    auto ring = [&](auto fast_tag) {
        const int S_ring = S - S % D;
        for (int s0 = 0; s0 < S_ring; s0 += D) {
#pragma unroll
            for (int d = 0; d < D; ++d) step(s0 + d, wb[d], fast_tag);
        }
#pragma unroll
        for (int d = 0; d < D; ++d)
            if (S_ring + d < S) step(S_ring + d, wb[d], fast_tag);
    };
    if (interior)
        ring(std::true_type{});
    else
        ring(std::false_type{});
    // Shifts beyond the halo: gather form, neighbour values from HBM.
    for (int s = 0; s < S && act; ++s) {
        const ShiftRec rc = read_shift(shl, s);
        if (shift_in_lds(rc)) continue;
        const T* wp = w_b + static_cast<int64_t>(s) * wstep;
        const int hp = wrap1(h + rc.dxm, H), hm = wrap1(h - rc.dxm, H);
        const int wp_ = wrap1(wq + rc.dym, W), wm_ = wrap1(wq - rc.dym, W);
        const uint32_t jp = static_cast<uint32_t>(hp) * W + wp_;
        const uint32_t jm = static_cast<uint32_t>(hm) * W + wm_;
        const int64_t ip = off + jp, im = off + jm;
        const bool okp = rc.inv && (rc.per || (in_range(h + rc.dx, H) && in_range(wq + rc.dy, W)));
        A xf[NC], ap[NC], bp[NC], fo;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            xf[c] = to_acc(x[ip + c * HW]);
            ap[c] = gDg[ip + c * HW];
            bp[c] = gLg[ip + c * HW] - ap[c] * Dg[ip + c * HW];
        }
        const A lp = LOGW ? log_key<A>(Lg[ip]) : Lim<A>::ex(-Lg[ip]);
        const A wv = fwd_kept(rc, h, wq, H, W) ? to_acc(wp[own]) : masked_key<A, LOGW>();
        const A g = terms(wv, xf, lp, ap, bp, okp, fo);
        g_b[static_cast<int64_t>(s) * wstep + own] = from_acc<T>(g);
        // x-gradient term from o = (q - s) mod: f(w_s[o], L[o]) gD[o]
        const A lm = LOGW ? Lg[im] : Lim<A>::ex(-Lg[im]);
        const A wo = fwd_kept_src(rc, h, wq, H, W) ? to_acc(wp[jm]) : masked_key<A, LOGW>();
        const A f = frac_tile<A, LOGW>(wo, lm);
#pragma unroll
        for (int c = 0; c < NC; ++c) gxa[c] = fma_acc(f, gDg[im + c * HW], gxa[c]);
    }
    __syncthreads();
    if (act) {
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const A v = gxa[c] + mg[c * G::TILE + li];
            const int64_t o = off + c * HW + own;
            if (gxp != nullptr)
                gxp[o] = v;
            else
                gx[o] = from_acc<T>(v);
        }
    }
    if (R == 0) return;
    const int n = spill_count(ti.th, ti.tw, R);
    const int64_t per_plane = static_cast<int64_t>(tg.ntw) * tg.nth;
    const int64_t tile = t - ti.bc * per_plane;
    for (int e = threadIdx.x; e < n; e += blockDim.x) {
        int i, j;
        spill_coords(e, ti.th, ti.tw, R, i, j);
        const int l = (i + HALO) * G::PITCH + j + HALO;
#pragma unroll
        for (int c = 0; c < NC; ++c)
            spill[((ti.bc * NC + c) * per_plane + tile) * G::SPILL + e] = mg[c * G::TILE + l];
    }
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------
constexpr size_t kNLdsLimit = 64 * 1024;

template <int VEC>
static size_t nfwd_lds(int S, size_t ab) {
    return shift_lds_bytes(S) + static_cast<size_t>(NGeo<VEC>::LH) * NGeo<VEC>::LW * ab;
}
template <int VEC>
static size_t nbwd_lds(int S, size_t ab) {
    return shift_lds_bytes(S) + 5 * static_cast<size_t>(NGeo<VEC>::LH) * NGeo<VEC>::LW * ab;
}

template <typename T>
static size_t n_lds(int v, int S, bool bwd) {
    const size_t ab = sizeof(acc_t<T>);
    switch (v) {
        case 8: return bwd ? nbwd_lds<8>(S, ab) : nfwd_lds<8>(S, ab);
        case 4: return bwd ? nbwd_lds<4>(S, ab) : nfwd_lds<4>(S, ab);
        case 2: return bwd ? nbwd_lds<2>(S, ab) : nfwd_lds<2>(S, ab);
        default: return bwd ? nbwd_lds<1>(S, ab) : nfwd_lds<1>(S, ab);
    }
}

template <typename T>
static int n_pick_vec(int W, std::initializer_list<const void*> ptrs, int S, bool bwd) {
    for (int v = 16 / static_cast<int>(sizeof(T)); v > 1; v /= 2) {
        if (W % v) continue;
        bool ok = true;
        for (const void* p : ptrs) ok = ok && nsh_host::aligned(p, v * sizeof(T));
        if (ok && n_lds<T>(v, S, bwd) <= kNLdsLimit) return v;
    }
    return 1;
}

struct NDims {
    int S, B, C, H, W;
    int codes = 0;  // kCodesRows / kCodesSharedW (from NSH_SHIFT_CODES, NSH_SHARED_WEIGHTS)
    bool narrow = false;  // NSH_NARROW_HALO: every row within 6 pixels (a hint)
    bool wide = false;    // NSH_WIDE_HALO: the radius lies in 9..16 (a hint)
};

template <typename T, int VEC, bool LOGW>
static int n_launch_fwd(const void* x, const void* w, const int64_t* sh, NDims d, void* D, void* L,
                        int* weights_ok, hipStream_t st) {
    using G = NGeo<VEC>;
    const int ntw = static_cast<int>(nsh_host::ceil_div(d.W, G::TW));
    const int nth = static_cast<int>(nsh_host::ceil_div(d.H, G::TH));
    const int64_t tiles = static_cast<int64_t>(d.B) * d.C * ntw * nth;
    const int64_t step = static_cast<int64_t>(d.B) * d.C * d.H * d.W;
    hipLaunchKernelGGL((normalized_fwd_kernel<T, VEC, LOGW>), dim3(static_cast<unsigned>(tiles)),
                       dim3(kThreads), n_lds<T>(VEC, d.S, false), st, static_cast<const T*>(x),
                       static_cast<const T*>(w), sh, d.S, d.codes, d.C, d.H, d.W, ntw, nth, step,
                       static_cast<acc_t<T>*>(D), static_cast<acc_t<T>*>(L), weights_ok);
    return nsh_host::check_launch("normalized_accumulate_uz_forward");
}

template <typename T, int VEC, bool LOGW>
static int n_launch_bwd(const void* x, const void* w, const void* D, const void* L, const void* gD,
                        const void* gL, const int64_t* sh, NDims d, void* gx, void* gw,
                        hipStream_t st) {
    using G = NGeo<VEC>;
    using A = acc_t<T>;
    const int ntw = static_cast<int>(nsh_host::ceil_div(d.W, G::TW));
    const int nth = static_cast<int>(nsh_host::ceil_div(d.H, G::TH));
    const int64_t tiles = static_cast<int64_t>(d.B) * d.C * ntw * nth;
    const int64_t step = static_cast<int64_t>(d.B) * d.C * d.H * d.W;
    hipLaunchKernelGGL((normalized_bwd_kernel<T, VEC, LOGW>), dim3(static_cast<unsigned>(tiles)),
                       dim3(kThreads), n_lds<T>(VEC, d.S, true), st, static_cast<const T*>(x),
                       static_cast<const T*>(w), static_cast<const A*>(D), static_cast<const A*>(L),
                       static_cast<const A*>(gD), static_cast<const A*>(gL), sh, d.S, d.codes, d.C, d.H,
                       d.W, ntw, nth, step, static_cast<T*>(gx), static_cast<T*>(gw));
    return nsh_host::check_launch("normalized_accumulate_uz_backward");
}

// ---- scatter path -------------------------------------------------------
// Tiles of 16 lanes x VEC pixels (4; 2 for fp64) across, 32 rows down
// (512-lane workgroups; the fp32 passes take 32 lanes, 128 x 32 tiles): the
// forward keeps four LDS arrays (x and the three state windows), the
// backward five (x, L or E, alpha, beta, window).  Weight prefetch depth 2,
// except the fp64 backward: four shifts in flight (c3 fp64 0.226 -> 0.213
// ms); depth 3 or 4 makes the fp32 passes and every forward 1-3% slower.
// fp32 forward: 128 x 32 tiles with nontemporal weight loads, c3 positive
// 0.329 -> 0.322 ms; the 16-bit forward stays on 64 x 32 tiles with plain
// loads (c2 logits 0.150 ms against 0.154 ms wide, 0.159 ms wide and
// nontemporal).  fp32 backward: 32 lanes per row (128 x 32 tiles, one
// workgroup per CU): c3 positive 0.690 -> 0.666 ms; the 16-bit backward
// stays at 16 (c2 logits 0.236 ms against 0.254 ms on the wide tiles).
// Variants:
//  * kNNarrow: the fp64 backward on a 6-pixel border (NSH_NARROW_HALO): 32 x 16
//    tiles, three 256-lane workgroups per CU (the c3 fp64 shape's 768 tiles in
//    one round; 32 x 16 on the 8-pixel border, two workgroups per CU and 1.5
//    rounds, measured no faster than 32 x 32; 1-pixel lanes on the narrow
//    border, 24 waves per CU: no faster);
//  * kNSlim: fp32 on 64 x 32 tiles for images of at most 64 columns, where half
//    the lanes of a 128-wide tile would idle;
//  * kNWide: a 16-pixel border for tables of radius 9..16 (NSH_WIDE_HALO; fp32
//    and 16-bit): 64 x 32 tiles of 1024 lanes, 2 pixels each (one workgroup per
//    CU: forward 98 KB of LDS plus the table, backward 143 KB).  On the 8-pixel
//    border such tables' far rows take the gather loop, one row's loads at a
//    time (half-plane R = 10, 221 rows, fp32: 1024^2 forward 524 -> 350 us,
//    backward 1115 -> 471 us; 3 x 792^2 1308 -> 647 and 2886 -> 1108).  Bound by
//    the loop's instructions and LDS latency at 16 waves per CU, not by the
//    stream (fp16 takes as long): 4-pixel lanes, half the waves, 396 and 538 us.
enum { kNBase = 0, kNNarrow = 1, kNSlim = 2, kNWide = 3 };
constexpr int kNSlimWidth = 64;
template <typename T, bool BWD, int VAR = kNBase>
struct NScatterCfg {
    static constexpr bool NARROW = VAR == kNNarrow, SLIM = VAR == kNSlim, WIDE = VAR == kNWide;
    static_assert(!SLIM || sizeof(T) == 4, "the other types' tiles are 64 wide or less");
    static_assert(!NARROW || (BWD && sizeof(T) == 8), "the narrow border serves the fp64 backward");
    static_assert(!WIDE || sizeof(T) <= 4, "fp64 tiles do not fit a 16-pixel border");
    static constexpr int VEC = (sizeof(T) == 8 || WIDE) ? 2 : 4;
    static constexpr int TPR = ((sizeof(T) == 4 && !SLIM) || WIDE) ? 32 : kTPR;
    // fp64 forward: 32 x 16 tiles (twice the workgroups; c3 0.083 -> 0.080 ms)
    static constexpr int ROWS = ((!BWD || NARROW) && sizeof(T) == 8) ? 16 : 32;
    static constexpr int HALO = NARROW ? 6 : (WIDE ? 16 : kRmax);
    // prefetch depth: 4 for the fp64 backward on the 8-pixel border, 2 on
    // the narrow one (c3 fp64 0.189 ms at 4, 0.181 at 2, 0.191 at 6); on the
    // wide one 2 forward and 4 backward (1024^2 R = 10 fp32: forward 350 us at
    // 2, 373 at 4, backward 496 and 471, 460 at 8)
    static constexpr int D = (BWD && (WIDE || (sizeof(T) == 8 && !NARROW))) ? 4 : 2;
    // register budget: a 1024-lane workgroup holds a CU alone (its LDS), so
    // four waves per SIMD; smaller ones two workgroups per CU, the narrow
    // border's three
    static constexpr int WPE = NARROW ? 3
                                      : (TPR * ROWS >= 1024 ? 4 : kScatterWavesPerEU<TPR * ROWS>);
    using G = std::conditional_t<BWD, NTileGeo<VEC, ROWS, TPR, HALO, (HALO < kRmax)>,
                                 NTileGeo<VEC, ROWS, TPR, HALO>>;
};

constexpr size_t kNScatterLds = 160 * 1024 - 1024;
constexpr int64_t kNHeader = 256;
// A gradient this small stays in the 256 MB Infinity Cache, which joins the
// streamed parts of a line (4 x 250^2 fp64 R = 6 backward 84 us, plain 100).
constexpr int64_t kNCachedBytes = int64_t(192) << 20;
// Smaller images are mostly border; the gather kernels read them from the
// caches.  From here on every tile is at least kRmax wide and high
// (nsh_host::tile_grid), so a window's border reaches only adjacent tiles
// (with one tile in a direction, the tile itself, as on a torus).
constexpr int kNScatterMinSide = 32;

struct NPlan {
    bool ok = false;
    int var = kNBase;
    int spill = 0, ring = 0;
    TileGrid grid{};
    int64_t tiles = 0, spill_bytes = 0, part_bytes = 0, total = 0;
    size_t lds = 0;
};

static int64_t n_align256(int64_t b) { return (b + 255) / 256 * 256; }

template <typename T, bool BWD, int VAR = kNBase>
static NPlan n_plan_cfg(const NDims& d) {
    using Cfg = NScatterCfg<T, BWD, VAR>;
    using G = typename Cfg::G;
    constexpr bool bwd = BWD;
    const int64_t ab = sizeof(acc_t<T>);
    NPlan p;
    p.var = VAR;
    constexpr int kReach = VAR == kNWide ? 16 : kRmax;  // the tables' largest radius
    p.grid = nsh_host::tile_grid(d.H, d.W, G::TH, G::TW, kReach);
    p.tiles = static_cast<int64_t>(d.B) * d.C * p.grid.ntw * p.grid.nth;
    p.lds = shift_lds_bytes(d.S) +
            (bwd ? 5 : 4) * static_cast<size_t>(G::TILE) * ab;
    p.spill = G::SPILL;
    p.ring = G::RING;
    p.ok = p.grid.narrow >= kReach && d.H >= kNScatterMinSide && d.W >= kNScatterMinSide &&
           p.lds <= kNScatterLds;
    p.spill_bytes = n_align256((bwd ? 1 : 3) * p.tiles * p.spill * ab);
    if (bwd)
        p.part_bytes = sizeof(T) < sizeof(acc_t<T>)
                           ? n_align256(static_cast<int64_t>(d.B) * d.C * d.H * d.W * ab)
                           : 0;
    else
        p.part_bytes = n_align256(3 * p.tiles * p.ring * ab);
    p.total = kNHeader + p.spill_bytes + p.part_bytes;
    return p;
}

// The plan: the variant that the caller's hint or the width asks for, where
// it applies and `hints` allows it, else the base one.
template <typename T, bool BWD>
static NPlan n_plan(const NDims& d, bool hints = true) {
    if (hints) {
        if constexpr (sizeof(T) == 8 && BWD) {
            if (d.narrow) {
                const NPlan p = n_plan_cfg<T, true, kNNarrow>(d);
                if (p.ok) return p;
            }
        }
        if constexpr (sizeof(T) <= 4) {
            if (d.wide) {
                const NPlan p = n_plan_cfg<T, BWD, kNWide>(d);
                if (p.ok) return p;
            }
        }
    }
    if constexpr (sizeof(T) == 4)
        if (d.W <= kNSlimWidth) return n_plan_cfg<T, BWD, kNSlim>(d);
    return n_plan_cfg<T, BWD>(d);
}

static bool n_scatter_disabled() {
    static const bool off = [] {
        const char* e = getenv("NSH_NORM_SCATTER");
        return e != nullptr && e[0] == '0';
    }();
    return off;
}

template <typename T>
static bool n_use_scatter(const NPlan& p, void* ws, int64_t ws_bytes) {
    return ws != nullptr && !n_scatter_disabled() && p.ok && ws_bytes >= p.total &&
           nsh_host::aligned(ws, 256);
}

// NH > 1: w is a head stack (S*B, NH, H, W) mixed by mix (C, NH) in the
// kernel's weight load.
template <typename T, bool LOGW, int NH, int VAR>
static int n_scatter_fwd_cfg(const void* x, const void* w, const int64_t* sh, NDims d, void* D,
                         void* L, const NPlan& p, void* ws, int* weights_ok, hipStream_t st,
                         const acc_t<T>* mix = nullptr) {
    using Cfg = NScatterCfg<T, false, VAR>;
    using A = acc_t<T>;
    constexpr int V = Cfg::VEC, TPR = Cfg::TPR, RW = Cfg::ROWS;
    char* base = static_cast<char*>(ws);
    int* hdr = reinterpret_cast<int*>(base);
    A* spill = reinterpret_cast<A*>(base + kNHeader);
    A* part = reinterpret_cast<A*>(base + kNHeader + p.spill_bytes);
    const int64_t step = static_cast<int64_t>(d.B) * (NH > 1 ? NH : d.C) * d.H * d.W;
    // Four heads' ring slots take 32 registers a shift ahead: at depth 2 the
    // kernel spilled 17 to 27 of them (4 heads, C = 3, R = 5 512^2 fp32 160 -> 146
    // us, R = 7 1024^2 fp16 663 -> 614).
    constexpr int D_ = NH == 4 ? 1 : Cfg::D;
    hipLaunchKernelGGL((normalized_fwd_scatter_kernel<T, V, TPR, RW, D_, LOGW, Cfg::WPE, NH,
                                                      Cfg::HALO>),
                       dim3(static_cast<unsigned>(p.tiles)), dim3(TPR * RW), p.lds, st,
                       static_cast<const T*>(x), static_cast<const T*>(w), sh, d.S, d.codes, d.C, d.H, d.W,
                       p.grid, step, static_cast<A*>(D), static_cast<A*>(L), hdr, spill, part,
                       p.ring, p.tiles, mix, weights_ok);
    if (int rc = nsh_host::check_launch("normalized_accumulate_uz_forward")) return rc;
    hipLaunchKernelGGL((normalized_fixup_kernel<A, LOGW>), dim3(static_cast<unsigned>(p.tiles)),
                       dim3(256), 0, st, d.H, d.W, RW, TPR * V, p.grid, p.spill, p.ring,
                       static_cast<const int*>(hdr), static_cast<const A*>(spill),
                       static_cast<const A*>(part), p.tiles, static_cast<A*>(D),
                       static_cast<A*>(L));
    return nsh_host::check_launch("normalized_accumulate_uz_forward (fix-up)");
}

template <typename T, bool LOGW, int NH = 1>
static int n_scatter_fwd(const void* x, const void* w, const int64_t* sh, NDims d, void* D,
                         void* L, const NPlan& p, void* ws, int* weights_ok, hipStream_t st,
                         const acc_t<T>* mix = nullptr) {
    if constexpr (sizeof(T) == 4)
        if (p.var == kNSlim)
            return n_scatter_fwd_cfg<T, LOGW, NH, kNSlim>(x, w, sh, d, D, L, p, ws, weights_ok,
                                                          st, mix);
    if constexpr (sizeof(T) <= 4)
        if (p.var == kNWide)
            return n_scatter_fwd_cfg<T, LOGW, NH, kNWide>(x, w, sh, d, D, L, p, ws, weights_ok,
                                                          st, mix);
    return n_scatter_fwd_cfg<T, LOGW, NH, kNBase>(x, w, sh, d, D, L, p, ws, weights_ok, st, mix);
}

template <typename T, bool LOGW, int VAR>
static int n_scatter_bwd_cfg(const void* x, const void* w, const void* D, const void* L,
                             const void* gD, const void* gL, const int64_t* sh, NDims d, void* gx,
                             void* gw, const NPlan& p, void* ws, hipStream_t st) {
    using Cfg = NScatterCfg<T, true, VAR>;
    using A = acc_t<T>;
    constexpr int V = Cfg::VEC, TPR = Cfg::TPR, RW = Cfg::ROWS;
    char* base = static_cast<char*>(ws);
    int* hdr = reinterpret_cast<int*>(base);
    A* spill = reinterpret_cast<A*>(base + kNHeader);
    A* part = p.part_bytes ? reinterpret_cast<A*>(base + kNHeader + p.spill_bytes) : nullptr;
    const int64_t step = static_cast<int64_t>(d.B) * d.C * d.H * d.W;
    // Contiguous 16-byte lanes where the row length and the pointers allow.
    const size_t vb = static_cast<size_t>(V) * sizeof(T);
    constexpr bool kContig = V == 4 || VAR == kNWide;
    const bool contig = kContig && d.W % V == 0 && nsh_host::aligned(x, vb) &&
                        nsh_host::aligned(w, vb) && nsh_host::aligned(gw, vb);
    const bool lines = static_cast<int64_t>(d.W) * sizeof(T) % 128 == 0;
    const bool small = step * d.S * static_cast<int64_t>(sizeof(T)) < kNCachedBytes;
    const bool stream = lines || (contig && (sizeof(T) == 4 || small)) || (!kContig && small);
    auto go = [&](auto contig_tag, auto nts_tag) {
        hipLaunchKernelGGL((normalized_bwd_scatter_kernel<T, V, TPR, RW, Cfg::D, LOGW,
                                                          decltype(contig_tag)::value,
                                                          decltype(nts_tag)::value, Cfg::WPE,
                                                          Cfg::HALO>),
                           dim3(static_cast<unsigned>(p.tiles)), dim3(TPR * RW), p.lds, st,
                           static_cast<const T*>(x), static_cast<const T*>(w),
                           static_cast<const A*>(D), static_cast<const A*>(L),
                           static_cast<const A*>(gD), static_cast<const A*>(gL), sh, d.S, d.codes,
                           d.C, d.H, d.W, p.grid, step, static_cast<T*>(gx), part,
                           static_cast<T*>(gw), hdr, spill);
    };
    if constexpr (kContig) {
        if (contig && stream)
            go(std::true_type{}, std::true_type{});
        else if (contig)
            go(std::true_type{}, std::false_type{});
        else
            go(std::false_type{}, std::false_type{});
    } else {
        if (stream)
            go(std::false_type{}, std::true_type{});
        else
            go(std::false_type{}, std::false_type{});
    }
    if (int rc = nsh_host::check_launch("normalized_accumulate_uz_backward")) return rc;
    constexpr bool kPart = sizeof(T) < sizeof(A);
    hipLaunchKernelGGL((spill_fixup_kernel<T, A, 1, kPart>), dim3(static_cast<unsigned>(p.tiles)),
                       dim3(256), 0, st, d.H, d.W, RW, TPR * V, p.grid, p.spill,
                       static_cast<const int*>(hdr), static_cast<const A*>(spill), p.tiles,
                       static_cast<const A*>(part), static_cast<T*>(gx), static_cast<T*>(nullptr));
    return nsh_host::check_launch("normalized_accumulate_uz_backward (fix-up)");
}

template <typename T, bool LOGW>
static int n_scatter_bwd(const void* x, const void* w, const void* D, const void* L,
                         const void* gD, const void* gL, const int64_t* sh, NDims d, void* gx,
                         void* gw, const NPlan& p, void* ws, hipStream_t st) {
    if constexpr (sizeof(T) == 8)
        if (p.var == kNNarrow)
            return n_scatter_bwd_cfg<T, LOGW, kNNarrow>(x, w, D, L, gD, gL, sh, d, gx, gw, p, ws,
                                                        st);
    if constexpr (sizeof(T) == 4)
        if (p.var == kNSlim)
            return n_scatter_bwd_cfg<T, LOGW, kNSlim>(x, w, D, L, gD, gL, sh, d, gx, gw, p, ws, st);
    if constexpr (sizeof(T) <= 4)
        if (p.var == kNWide)
            return n_scatter_bwd_cfg<T, LOGW, kNWide>(x, w, D, L, gD, gL, sh, d, gx, gw, p, ws, st);
    return n_scatter_bwd_cfg<T, LOGW, kNBase>(x, w, D, L, gD, gL, sh, d, gx, gw, p, ws, st);
}

// Either plan may run (the base one when the workspace is too small for the
// hinted one): the larger of the two.
template <typename T, bool BWD>
static int64_t n_workspace(const NDims& d) {
    const NPlan p = n_plan<T, BWD>(d, false);
    const NPlan q = n_plan<T, BWD>(d);
    return std::max(p.ok ? p.total : 0, q.ok ? q.total : 0);
}
template <typename T>
static int64_t n_workspace(const NDims& d, bool bwd) {
    return bwd ? n_workspace<T, true>(d) : n_workspace<T, false>(d);
}

// Whether the gather kernels beat the tiles that would serve a call: rows that
// take no vectors of 4 on few workgroups of the gather kernels (16 rows x 16
// vectors, 256 lanes), whose one- and two-pixel lanes walk the table faster
// than the tiles' four, as long as all of them run at once; and forwards of
// tables of a few rows, whose spilled border and fix-up cost as much as the
// rows.  In us, tiles and gather kernels, or the ratio of the two:
//  * fp32, odd rows: 137 x 73 R = 4 forward 58 / 25, backward 57 / 35; window
//    R = 5 133^2 77 / 36 and 142 / 84; at 1024 workgroups R = 5 1.16 to 1.45, at
//    1444 0.97 to 1.28, at 2048 0.8;
//  * fp32, W % 4 = 2: 1.0 to 1.7 at 330 workgroups, 0.8 to 1.1 at 780 (in up to
//    96 columns a third of the gather's lanes idle: R = 8 3 x 1023 x 38 122 / 175);
//  * 16-bit, odd rows: forward 1.0 to 1.5 at 720, backward 0.9 to 1.2 at 1024
//    (R = 8 0.9 at 620 and 1000); W % 4 = 2: R = 3 1.0 to 1.4 at 510, R = 5 0.9 to
//    1.2 at 360, R = 7 0.5 to 0.8;
//  * on a wide border the tiles' lanes hold two pixels and win sooner (R = 9
//    36 x 59 131 / 100; R = 10 953 x 97, 1260 workgroups, 170 / 250);
//  * fp64, forward: R = 1 192 x 35 x 154 86 / 34, odd rows R = 3 1.0 to 1.3 at
//    1024, window R = 4 53 x 71 36 / 28;
//  * few rows: fp32 R = 1 96 x 128 20 / 14, R = 2 3 x 160^2 28 / 22; fp16 R = 1 64 x
//    259 x 134 60 / 39;
//  * 128-wide fp32 tiles mostly beyond a narrow image: R = 3 192 x 48 x 129
//    121 / 94.
template <typename T, bool BWD>
static bool n_gather_instead(const NDims& d) {
    const int vec = d.W % 2 ? 1 : (d.W % 4 ? 2 : 4);
    const int64_t blocks = static_cast<int64_t>(d.B) * d.C * nsh_host::ceil_div(d.H, 16) *
                           nsh_host::ceil_div(d.W, 16 * vec);
    const bool few = !BWD && d.S <= 13;
    int most;  // workgroups per compute unit up to which the gather kernels win
    if (sizeof(T) == 8) {
        most = d.S <= 25 ? 4 : (d.S <= 81 ? 1 : 0);
        most = BWD || vec > 1 ? 0 : most;
        if (few) return true;
    } else if (vec == 1) {
        if (few && d.S <= 5) return true;
        const int half = BWD ? 4 : 3;  // 16-bit
        most = sizeof(T) == 4 || d.S <= 25 ? 5 : (d.S <= 81 ? half : half - 1);
        most = d.wide ? 1 : (few ? 8 : most);
    } else if (vec == 2) {
        if (few && (sizeof(T) == 4 || d.S <= 5)) return true;
        const int half = d.S <= 25 ? 2 : (d.S <= 61 ? 1 : 0);  // 16-bit
        most = d.wide || d.W <= 96 ? 0 : (sizeof(T) == 4 ? 2 : half);
    } else {
        most = few && sizeof(T) == 4 && d.W > 64 ? 2 : 0;
    }
    if (!BWD && sizeof(T) == 4 && vec < 4 && d.S <= 25 && d.W > 64 &&
        5 * nsh_host::ceil_div(d.W, 128) * 128 >= 8 * d.W)
        return true;
    return most > 0 && blocks <= most * static_cast<int64_t>(nsh_host::compute_units());
}

// The plan that a call's workspace allows (p.ok is false if none).
template <typename T, bool BWD>
static NPlan n_usable_plan(const NDims& d, void* ws, int64_t ws_bytes) {
    NPlan p = n_plan<T, BWD>(d);
    if (!n_use_scatter<T>(p, ws, ws_bytes)) p = n_plan<T, BWD>(d, false);
    p.ok = n_use_scatter<T>(p, ws, ws_bytes);
    return p;
}

template <typename T, bool LOGW>
static int n_run_fwd(const void* x, const void* w, const int64_t* sh, NDims d, void* D, void* L,
                     void* ws, int64_t ws_bytes, int* weights_ok, hipStream_t st) {
    const NPlan p = n_usable_plan<T, false>(d, ws, ws_bytes);
    if (p.ok && !n_gather_instead<T, false>(d))
        return n_scatter_fwd<T, LOGW>(x, w, sh, d, D, L, p, ws, weights_ok, st);
    switch (n_pick_vec<T>(d.W, {x, w, D, L}, d.S, false)) {
        case 8: if constexpr (sizeof(T) == 2) return n_launch_fwd<T, 8, LOGW>(x, w, sh, d, D, L, weights_ok, st); break;
        case 4: if constexpr (sizeof(T) <= 4) return n_launch_fwd<T, 4, LOGW>(x, w, sh, d, D, L, weights_ok, st); break;
        case 2: return n_launch_fwd<T, 2, LOGW>(x, w, sh, d, D, L, weights_ok, st);
        default: break;
    }
    return n_launch_fwd<T, 1, LOGW>(x, w, sh, d, D, L, weights_ok, st);
}

template <typename T, bool LOGW>
static int n_run_bwd(const void* x, const void* w, const void* D, const void* L, const void* gD,
                     const void* gL, const int64_t* sh, NDims d, void* gx, void* gw, void* ws,
                     int64_t ws_bytes, hipStream_t st) {
    const NPlan p = n_usable_plan<T, true>(d, ws, ws_bytes);
    if (p.ok && !n_gather_instead<T, true>(d))
        return n_scatter_bwd<T, LOGW>(x, w, D, L, gD, gL, sh, d, gx, gw, p, ws, st);
    switch (n_pick_vec<T>(d.W, {x, w, D, L, gD, gL, gx, gw}, d.S, true)) {
        case 8: if constexpr (sizeof(T) == 2) return n_launch_bwd<T, 8, LOGW>(x, w, D, L, gD, gL, sh, d, gx, gw, st); break;
        case 4: if constexpr (sizeof(T) <= 4) return n_launch_bwd<T, 4, LOGW>(x, w, D, L, gD, gL, sh, d, gx, gw, st); break;
        case 2: return n_launch_bwd<T, 2, LOGW>(x, w, D, L, gD, gL, sh, d, gx, gw, st);
        default: break;
    }
    return n_launch_bwd<T, 1, LOGW>(x, w, D, L, gD, gL, sh, d, gx, gw, st);
}

// The shared-weight backward with the summed gradient: two or three channels
// of fp32 or 16-bit type on images the tiles serve.
struct NShPlan {
    bool ok = false;
    TileGrid grid{};
    int64_t tiles = 0, spill_bytes = 0, part_bytes = 0, total = 0;
    size_t lds = 0;
};

template <typename T>
static NShPlan n_shared_plan(const NDims& d) {
    using G = SGeo<1, kNShRows, kNShTpr>;
    const int64_t ab = sizeof(acc_t<T>);
    NShPlan p;
    p.grid = nsh_host::tile_grid(d.H, d.W, G::TH, G::TW);
    p.tiles = static_cast<int64_t>(d.B) * p.grid.ntw * p.grid.nth;  // per channel
    p.lds = shift_lds_bytes(d.S) + (4 * d.C + 1) * static_cast<size_t>(G::TILE) * ab;
    p.ok = sizeof(T) <= 4 && (d.C == 2 || d.C == 3) && p.grid.narrow >= kRmax &&
           d.H >= kNScatterMinSide && d.W >= kNScatterMinSide && p.lds <= kNScatterLds;
    p.spill_bytes = n_align256(p.tiles * d.C * G::SPILL * ab);
    p.part_bytes = sizeof(T) < sizeof(acc_t<T>)
                       ? n_align256(static_cast<int64_t>(d.B) * d.C * d.H * d.W * ab)
                       : 0;
    p.total = kNHeader + p.spill_bytes + p.part_bytes;
    return p;
}

template <typename T, bool LOGW>
static int n_run_bwd_shared(const void* x, const void* w, const void* D, const void* L,
                            const void* gD, const void* gL, const int64_t* sh, NDims d, void* gx,
                            void* gw, void* ws, int64_t ws_bytes, hipStream_t st) {
    using A = acc_t<T>;
    using G = SGeo<1, kNShRows, kNShTpr>;
    const NShPlan p = n_shared_plan<T>(d);
    if (!p.ok || n_scatter_disabled() || ws == nullptr || ws_bytes < p.total ||
        !nsh_host::aligned(ws, 256))
        return nsh_host::fail(NSH_ERR_UNSUPPORTED,
                              "normalized_accumulate_uz_backward_shared: shape or workspace not "
                              "served");
    char* base = static_cast<char*>(ws);
    int* hdr = reinterpret_cast<int*>(base);
    A* spill = reinterpret_cast<A*>(base + kNHeader);
    A* part = p.part_bytes ? reinterpret_cast<A*>(base + kNHeader + p.spill_bytes) : nullptr;
    const int64_t wstep = static_cast<int64_t>(d.B) * d.H * d.W;
    auto go = [&](auto nc) {
        hipLaunchKernelGGL((normalized_bwd_shared_kernel<T, decltype(nc)::value, LOGW>),
                           dim3(static_cast<unsigned>(p.tiles)), dim3(G::THREADS), p.lds, st,
                           static_cast<const T*>(x), static_cast<const T*>(w),
                           static_cast<const A*>(D), static_cast<const A*>(L),
                           static_cast<const A*>(gD), static_cast<const A*>(gL), sh, d.S, d.codes,
                           d.H, d.W, p.grid, wstep, static_cast<T*>(gx), part,
                           static_cast<T*>(gw), hdr, spill);
    };
    if (d.C == 2)
        go(std::integral_constant<int, 2>{});
    else
        go(std::integral_constant<int, 3>{});
    if (int rc = nsh_host::check_launch("normalized_accumulate_uz_backward_shared")) return rc;
    constexpr bool kPart = sizeof(T) < sizeof(A);
    hipLaunchKernelGGL((spill_fixup_kernel<T, A, 1, kPart>),
                       dim3(static_cast<unsigned>(p.tiles * d.C)), dim3(256), 0, st, d.H, d.W,
                       G::TH, G::TW, p.grid, G::SPILL, static_cast<const int*>(hdr),
                       static_cast<const A*>(spill), p.tiles * d.C, static_cast<const A*>(part),
                       static_cast<T*>(gx), static_cast<T*>(nullptr));
    return nsh_host::check_launch("normalized_accumulate_uz_backward_shared (fix-up)");
}

}  // namespace nsh

using nsh_host::fail;

static int n_check(const char* op, int64_t S, int64_t B, int64_t C, int64_t H, int64_t W, int dtype,
                   nsh::NDims* d) {
    const int codes = nsh::dtype_codes(dtype);
    const bool narrow = (dtype & NSH_NARROW_HALO) != 0;
    const bool wide = (dtype & NSH_WIDE_HALO) != 0 && (dtype & NSH_WIDER_HALO) == 0;
    dtype &= ~NSH_DTYPE_FLAGS;
    if (S < 1 || S > 1024)
        return fail(NSH_ERR_INVALID, "%s: tree reduction requires 1 <= S <= 1024", op);
    if (B < 1 || C < 1 || H < 1 || W < 1)
        return fail(NSH_ERR_INVALID, "%s: empty tensor", op);
    if (dtype < NSH_DTYPE_FLOAT16 || dtype > NSH_DTYPE_FLOAT64)
        return fail(NSH_ERR_INVALID, "%s: unsupported dtype code %d", op, dtype);
    const int64_t es = dtype == NSH_DTYPE_FLOAT64 ? 8 : 4;
    if (H * W * es >= (int64_t(1) << 31))
        return fail(NSH_ERR_INVALID, "%s: one (b, c) plane must stay below 2^31 bytes", op);
    if (B * C > (int64_t(1) << 24)) return fail(NSH_ERR_INVALID, "%s: B*C too large", op);
    *d = nsh::NDims{static_cast<int>(S), static_cast<int>(B), static_cast<int>(C),
                    static_cast<int>(H), static_cast<int>(W), codes, narrow, wide};
    return NSH_OK;
}

#define NSH_DISPATCH_LOGW(T, FN, ...)                                   \
    (log_weights ? nsh::FN<T, true>(__VA_ARGS__) : nsh::FN<T, false>(__VA_ARGS__))

extern "C" int64_t nsh_normalized_workspace_bytes(int64_t S, int64_t B, int64_t C, int64_t H,
                                                  int64_t W, int dtype, int backward) {
    nsh::NDims d;
    if (n_check("normalized_accumulate_uz", S, B, C, H, W, dtype, &d) != NSH_OK) return -1;
    dtype &= ~NSH_DTYPE_FLAGS;
    const bool bwd = backward != 0;
    switch (dtype) {
        case NSH_DTYPE_FLOAT16: return nsh::n_workspace<nsh::f16>(d, bwd);
        case NSH_DTYPE_BFLOAT16: return nsh::n_workspace<nsh::bf16>(d, bwd);
        case NSH_DTYPE_FLOAT32: return nsh::n_workspace<float>(d, bwd);
        default: return nsh::n_workspace<double>(d, bwd);
    }
}

extern "C" int nsh_normalized_accumulate_uz_forward_checked(
    const void* x, const void* weights, const int64_t* shifts, int64_t S, int64_t B, int64_t C,
    int64_t H, int64_t W, int dtype, int log_weights, void* D, void* log_C, int* weights_ok,
    void* workspace, int64_t workspace_bytes, void* stream) {
    nsh::NDims d;
    if (int rc = n_check("normalized_accumulate_uz", S, B, C, H, W, dtype, &d)) return rc;
    dtype &= ~NSH_DTYPE_FLAGS;
    if (!x || !weights || !shifts || !D || !log_C)
        return fail(NSH_ERR_INVALID, "normalized_accumulate_uz: null pointer argument");
    hipStream_t st = static_cast<hipStream_t>(stream);
    void* ws = workspace;
    const int64_t nws = workspace ? workspace_bytes : 0;
    switch (dtype) {
        case NSH_DTYPE_FLOAT16: return NSH_DISPATCH_LOGW(nsh::f16, n_run_fwd, x, weights, shifts, d, D, log_C, ws, nws, weights_ok, st);
        case NSH_DTYPE_BFLOAT16: return NSH_DISPATCH_LOGW(nsh::bf16, n_run_fwd, x, weights, shifts, d, D, log_C, ws, nws, weights_ok, st);
        case NSH_DTYPE_FLOAT32: return NSH_DISPATCH_LOGW(float, n_run_fwd, x, weights, shifts, d, D, log_C, ws, nws, weights_ok, st);
        default: return NSH_DISPATCH_LOGW(double, n_run_fwd, x, weights, shifts, d, D, log_C, ws, nws, weights_ok, st);
    }
}

extern "C" int nsh_normalized_accumulate_uz_forward(const void* x, const void* weights,
                                                    const int64_t* shifts, int64_t S, int64_t B,
                                                    int64_t C, int64_t H, int64_t W, int dtype,
                                                    int log_weights, void* D, void* log_C,
                                                    void* workspace, int64_t workspace_bytes,
                                                    void* stream) {
    return nsh_normalized_accumulate_uz_forward_checked(x, weights, shifts, S, B, C, H, W, dtype,
                                                        log_weights, D, log_C, nullptr, workspace,
                                                        workspace_bytes, stream);
}

// Head mixing in the weight load: with a (C, heads) mix the scatter path
// only (the shapes the workspace plan serves), positive weights, no grad.
template <typename T>
static int n_run_fwd_mixed(const void* x, const void* hw, const void* mix, const int64_t* sh,
                           nsh::NDims d, int heads, void* D, void* L, void* ws, int64_t nws,
                           hipStream_t st) {
    using A = nsh::acc_t<T>;
    const nsh::NPlan p = nsh::n_usable_plan<T, false>(d, ws, nws);
    if (!p.ok)
        return fail(NSH_ERR_UNSUPPORTED,
                    "normalized_accumulate_uz_forward_mixed: shape or workspace not served by "
                    "the scatter path");
    const A* m = static_cast<const A*>(mix);
    switch (heads) {
        case 2: return nsh::n_scatter_fwd<T, false, 2>(x, hw, sh, d, D, L, p, ws, nullptr, st, m);
        case 3: return nsh::n_scatter_fwd<T, false, 3>(x, hw, sh, d, D, L, p, ws, nullptr, st, m);
        default: return nsh::n_scatter_fwd<T, false, 4>(x, hw, sh, d, D, L, p, ws, nullptr, st, m);
    }
}

extern "C" int nsh_normalized_accumulate_uz_forward_mixed(
    const void* x, const void* head_weights, const void* mix, const int64_t* shifts, int64_t S,
    int64_t B, int64_t C, int64_t H, int64_t W, int64_t heads, int dtype, void* D, void* log_C,
    void* workspace, int64_t workspace_bytes, void* stream) {
    nsh::NDims d;
    if (int rc = n_check("normalized_accumulate_uz_forward_mixed", S, B, C, H, W, dtype, &d))
        return rc;
    if (dtype & NSH_SHARED_WEIGHTS)
        return fail(NSH_ERR_INVALID,
                    "normalized_accumulate_uz_forward_mixed: shared weights do not apply to a "
                    "head stack");
    dtype &= ~NSH_DTYPE_FLAGS;
    if (!x || !head_weights || !mix || !shifts || !D || !log_C)
        return fail(NSH_ERR_INVALID, "normalized_accumulate_uz_forward_mixed: null pointer argument");
    if (heads < 2 || heads > 4)
        return fail(NSH_ERR_UNSUPPORTED,
                    "normalized_accumulate_uz_forward_mixed: %lld heads (2..4 are served)",
                    static_cast<long long>(heads));
    if (B * heads > (int64_t(1) << 24))
        return fail(NSH_ERR_INVALID, "normalized_accumulate_uz_forward_mixed: B*heads too large");
    hipStream_t st = static_cast<hipStream_t>(stream);
    const int64_t nws = workspace ? workspace_bytes : 0;
    const int h = static_cast<int>(heads);
    switch (dtype) {
        case NSH_DTYPE_FLOAT16: return n_run_fwd_mixed<nsh::f16>(x, head_weights, mix, shifts, d, h, D, log_C, workspace, nws, st);
        case NSH_DTYPE_BFLOAT16: return n_run_fwd_mixed<nsh::bf16>(x, head_weights, mix, shifts, d, h, D, log_C, workspace, nws, st);
        case NSH_DTYPE_FLOAT32: return n_run_fwd_mixed<float>(x, head_weights, mix, shifts, d, h, D, log_C, workspace, nws, st);
        default: return n_run_fwd_mixed<double>(x, head_weights, mix, shifts, d, h, D, log_C, workspace, nws, st);
    }
}

extern "C" int nsh_normalized_accumulate_uz_backward(const void* x, const void* weights,
                                                     const void* D, const void* log_C,
                                                     const void* grad_D, const void* grad_log_C,
                                                     const int64_t* shifts, int64_t S, int64_t B,
                                                     int64_t C, int64_t H, int64_t W, int dtype,
                                                     int log_weights, void* grad_x, void* grad_w,
                                                     void* workspace, int64_t workspace_bytes,
                                                     void* stream) {
    nsh::NDims d;
    if (int rc = n_check("normalized_accumulate_uz_backward", S, B, C, H, W, dtype, &d)) return rc;
    dtype &= ~NSH_DTYPE_FLAGS;
    if (!x || !weights || !D || !log_C || !grad_D || !grad_log_C || !shifts || !grad_x || !grad_w)
        return fail(NSH_ERR_INVALID, "normalized_accumulate_uz_backward: null pointer argument");
    hipStream_t st = static_cast<hipStream_t>(stream);
    void* ws = workspace;
    const int64_t nws = workspace ? workspace_bytes : 0;
    switch (dtype) {
        case NSH_DTYPE_FLOAT16:
            return NSH_DISPATCH_LOGW(nsh::f16, n_run_bwd, x, weights, D, log_C, grad_D, grad_log_C, shifts, d, grad_x, grad_w, ws, nws, st);
        case NSH_DTYPE_BFLOAT16:
            return NSH_DISPATCH_LOGW(nsh::bf16, n_run_bwd, x, weights, D, log_C, grad_D, grad_log_C, shifts, d, grad_x, grad_w, ws, nws, st);
        case NSH_DTYPE_FLOAT32:
            return NSH_DISPATCH_LOGW(float, n_run_bwd, x, weights, D, log_C, grad_D, grad_log_C, shifts, d, grad_x, grad_w, ws, nws, st);
        default:
            return NSH_DISPATCH_LOGW(double, n_run_bwd, x, weights, D, log_C, grad_D, grad_log_C, shifts, d, grad_x, grad_w, ws, nws, st);
    }
}

extern "C" int64_t nsh_normalized_shared_workspace_bytes(int64_t S, int64_t B, int64_t C, int64_t H,
                                                         int64_t W, int dtype) {
    nsh::NDims d;
    if (n_check("normalized_accumulate_uz_backward_shared", S, B, C, H, W, dtype, &d)) return -1;
    switch (dtype & ~NSH_DTYPE_FLAGS) {
        case NSH_DTYPE_FLOAT16:
        case NSH_DTYPE_BFLOAT16: {
            const nsh::NShPlan p = nsh::n_shared_plan<nsh::f16>(d);
            return p.ok ? p.total : 0;
        }
        case NSH_DTYPE_FLOAT32: {
            const nsh::NShPlan p = nsh::n_shared_plan<float>(d);
            return p.ok ? p.total : 0;
        }
        default: return 0;
    }
}

extern "C" int nsh_normalized_accumulate_uz_backward_shared(
    const void* x, const void* weights, const void* D, const void* log_C, const void* grad_D,
    const void* grad_log_C, const int64_t* shifts, int64_t S, int64_t B, int64_t C, int64_t H,
    int64_t W, int dtype, int log_weights, void* grad_x, void* grad_w, void* workspace,
    int64_t workspace_bytes, void* stream) {
    nsh::NDims d;
    if (int rc = n_check("normalized_accumulate_uz_backward_shared", S, B, C, H, W, dtype, &d))
        return rc;
    dtype &= ~NSH_DTYPE_FLAGS;
    if (!x || !weights || !D || !log_C || !grad_D || !grad_log_C || !shifts || !grad_x || !grad_w)
        return fail(NSH_ERR_INVALID,
                    "normalized_accumulate_uz_backward_shared: null pointer argument");
    hipStream_t st = static_cast<hipStream_t>(stream);
    const int64_t nws = workspace ? workspace_bytes : 0;
    switch (dtype) {
        case NSH_DTYPE_FLOAT16:
            return NSH_DISPATCH_LOGW(nsh::f16, n_run_bwd_shared, x, weights, D, log_C, grad_D, grad_log_C, shifts, d, grad_x, grad_w, workspace, nws, st);
        case NSH_DTYPE_BFLOAT16:
            return NSH_DISPATCH_LOGW(nsh::bf16, n_run_bwd_shared, x, weights, D, log_C, grad_D, grad_log_C, shifts, d, grad_x, grad_w, workspace, nws, st);
        case NSH_DTYPE_FLOAT32:
            return NSH_DISPATCH_LOGW(float, n_run_bwd_shared, x, weights, D, log_C, grad_D, grad_log_C, shifts, d, grad_x, grad_w, workspace, nws, st);
        default:
            return fail(NSH_ERR_UNSUPPORTED,
                        "normalized_accumulate_uz_backward_shared: fp64 is not served");
    }
}
