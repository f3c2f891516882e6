// The native Gated DeltaNet layer around K1 (reference: GatedDeltaNet.forward, Heimdall/heimdall/hibrit.py:159-184,
// causal_conv Heimdall/heimdall/kernels.py:29-37, l2norm hibrit.py:132-133, GatedNorm hibrit.py:118-129): the two
// memory-bound passes on either side of the delta rule, each one read and one write of its tensors.
//
// gdn_conv_inputs_kernel: from z = in_proj_qkv(x) (channels [q | k | v], C = 2 HK D + HV D) and the a / b gate
// projections, per token
//   y_c = SiLU(sum_j w[c][K-1-j] z[t-j][c])        causal depthwise conv, rows before the sequence start from the
//                                                   carried prefix (or zero)
//   q_h = D^-1/2 l2norm(y_q(h / r)), k_h = l2norm(y_k(h / r)), v_h = y_v(h)     for the HV value heads, r = HV / HK
//   beta = sigmoid(b), g = -exp(A_log) softplus(a + dt_bias)
// One unit = one q / k / v head of D channels, handled by D / 8 consecutive lanes of 8 channels each; the l2norm sum
// is a butterfly over those lanes. q and k are written once per value head that reads them (the
// reference's repeat_interleave), so the delta rule sees one key per state.
//
// gated_norm_kernel: out = w * RMSNorm(o) * SiLU(zg) per row of D; a bf16 layer keeps the reference's bf16 rounding
// points (o rounded to bf16, the normalised row rounded, the weight product rounded, then the SiLU product).
#include <type_traits>

#include "bf_common.h"
#include "bf_internal.h"

namespace bf {

namespace {

__device__ __forceinline__ float bf_round(float x) { return bf2f(f2bf(x)); }

__device__ __forceinline__ void unpack8(const uint4& u, float (&x)[8]) {
    const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        x[2 * i] = __uint_as_float(w[i] << 16);
        x[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
    }
}

__device__ __forceinline__ uint4 pack8(const float (&x)[8]) {
    return make_uint4(pack_bf16x2(x[0], x[1]), pack_bf16x2(x[2], x[3]), pack_bf16x2(x[4], x[5]),
                      pack_bf16x2(x[6], x[7]));
}

__device__ __forceinline__ void store8(void* base, long elem, int dtype, const float (&x)[8]) {
    if (dtype == DT_BF16) {
        *reinterpret_cast<uint4*>(reinterpret_cast<uint16_t*>(base) + elem) = pack8(x);
    } else {
        float4* p = reinterpret_cast<float4*>(reinterpret_cast<float*>(base) + elem);
        p[0] = make_float4(x[0], x[1], x[2], x[3]);
        p[1] = make_float4(x[4], x[5], x[6], x[7]);
    }
}

// sum over the LPU consecutive lanes of a unit (LPU a power of two <= 64)
template <int LPU>
__device__ __forceinline__ float unit_sum(float v) {
#pragma unroll
    for (int m = LPU / 2; m >= 1; m >>= 1) v += __shfl_xor(v, m);
    return v;
}

__device__ __forceinline__ float silu(float y) { return y / (1.f + __expf(-y)); }

// eight consecutive elements of a bf16 or fp32 row as fp32 (zero when !ok)
template <bool BF>
__device__ __forceinline__ void load8(const void* base, long elem, bool ok, float (&x)[8]) {
    if constexpr (BF) {
        unpack8(ok ? ld16(reinterpret_cast<const uint16_t*>(base) + elem) : zero16(), x);
    } else {
        const float4* p = reinterpret_cast<const float4*>(reinterpret_cast<const float*>(base) + elem);
        const float4 v0 = ok ? p[0] : make_float4(0.f, 0.f, 0.f, 0.f);
        const float4 v1 = ok ? p[1] : make_float4(0.f, 0.f, 0.f, 0.f);
        x[0] = v0.x; x[1] = v0.y; x[2] = v0.z; x[3] = v0.w; x[4] = v1.x; x[5] = v1.y; x[6] = v1.z; x[7] = v1.w;
    }
}

// channels c0 .. c0 + 7 of token n - j (rows before the sequence start come from the carried prefix, or are zero)
template <bool BF>
__device__ __forceinline__ void load_tap(const GdnInArgs& a, bool valid, long n, int j, long seq0, int seq, long C,
                                         int c0, float (&x)[8]) {
    const long p = n - j;
    if (p >= seq0) load8<BF>(a.z, p * a.z_st + c0, valid, x);
    else load8<BF>(a.prefix, ((long)seq * (a.K - 1) + (p - seq0 + a.K - 1)) * C + c0, valid && a.prefix, x);
}

}  // namespace

template <int D, bool BF>
__global__ __launch_bounds__(256) void gdn_conv_inputs_kernel(GdnInArgs a) {
    constexpr int LPU = D / 8;
    const int U = 2 * a.HK + a.HV;
    const long tid = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long unit = tid / LPU;
    const int s = (int)(tid % LPU);
    const bool valid = unit < a.n_tok * U;
    const long n = valid ? unit / U : 0;
    const int u = valid ? (int)(unit % U) : 0;

    // sequence of token n and its first token
    int lo = 0, hi = a.num_seqs;                          // cu[lo] <= n < cu[hi]
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (a.cu_seqlens[mid] <= n) lo = mid;
        else hi = mid;
    }
    const long seq0 = a.cu_seqlens[lo];

    const int kind = u < a.HK ? 0 : (u < 2 * a.HK ? 1 : 2);          // q, k, v
    const int head = kind == 0 ? u : (kind == 1 ? u - a.HK : u - 2 * a.HK);
    const long C = (long)(2 * a.HK + a.HV) * D;
    const int c0 = (kind == 0 ? head * D : (kind == 1 ? (a.HK + head) * D : 2 * a.HK * D + head * D)) + 8 * s;

    // tap j reads token n - j with weight column K - 1 - j; K = 4 (the models' conv width) takes each channel's
    // weights as one float4
    float y[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) y[e] = 0.f;
    if (a.K == 4) {
        float4 wc[8];
#pragma unroll
        for (int e = 0; e < 8; ++e)
            wc[e] = valid ? *reinterpret_cast<const float4*>(a.w + (long)(c0 + e) * 4) : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            float x[8];
            load_tap<BF>(a, valid, n, j, seq0, lo, C, c0, x);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float wj = j == 0 ? wc[e].w : (j == 1 ? wc[e].z : (j == 2 ? wc[e].y : wc[e].x));
                y[e] = fmaf(x[e], wj, y[e]);
            }
        }
    } else {
        for (int j = 0; j < a.K; ++j) {
            float x[8];
            load_tap<BF>(a, valid, n, j, seq0, lo, C, c0, x);
#pragma unroll
            for (int e = 0; e < 8; ++e) y[e] = fmaf(x[e], valid ? a.w[(long)(c0 + e) * a.K + (a.K - 1 - j)] : 0.f, y[e]);
        }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) y[e] = silu(y[e]);

    if (kind < 2) {
        float ss = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) ss += y[e] * y[e];
        ss = unit_sum<LPU>(ss);                           // every lane of the wave takes part
        const float f = rsqrtf(ss + a.eps) * (kind == 0 ? a.q_scale : 1.f);
#pragma unroll
        for (int e = 0; e < 8; ++e) y[e] *= f;
        if (!valid) return;
        const int r = a.HV / a.HK;
        void* dst = kind == 0 ? a.q : a.k;
        for (int rr = 0; rr < r; ++rr) store8(dst, (n * a.HV + head * r + rr) * D + 8 * s, a.out_dtype, y);
    } else {
        if (!valid) return;
        store8(a.v, (n * a.HV + head) * D + 8 * s, a.out_dtype, y);
        if (s == 0) {
            const long i = n * a.HV + head;
            const float x = a.a[i] + a.dt_bias[head];
            const float sp = x > 20.f ? x : log1pf(__expf(x));   // softplus with torch's default threshold
            a.g[i] = -__expf(a.A_log[head]) * sp;
            a.beta[i] = 1.f / (1.f + __expf(-a.b[i]));
        }
    }
}

// Conv width K = 4 (the models'): a thread keeps one unit's 8 channels over a block of CT consecutive tokens, with
// the channels' weights and the previous three rows in registers, so z is read once and the weights once per block
// (the per-token kernel above re-reads 4 rows and 128 bytes of weights for every 16 bytes of output).
// The outputs may alias z as far as the compiler knows, so a load of z is never moved above an earlier store: the
// rows of CP tokens are therefore loaded together before the group's stores, and the gates of the block's tokens are
// computed first, spread over the unit's lanes (computed per token by one lane, their loads put a second memory
// round trip into every token's chain). Measured on 4 packed sequences {8192, 16384, 24576, 16384}, H = 32, D = 128,
// bf16: 915-999 us before, 770-880 us with the gates first, 740-820 us with 4-row groups and 64-token blocks (2-row
// groups 870 us; 8-row groups 820-850 us at 155 VGPRs; streaming z loads or output stores within noise).
// A block takes 64 tokens when that gives the chip enough blocks, else fewer (conv_block): a decode step of 32
// sequences is 6 blocks of 64 tokens, 49 us of serial rows, and 48 blocks of 4 tokens (H = 32, D = 128).
constexpr int CP = 4;
static int conv_block(long n_tok, int ugroups) {
    int ct = 64;
    while (ct > CP && (n_tok + ct - 1) / ct * ugroups < 512) ct /= 2;
    return ct;
}

template <int D, bool BF>
__global__ __launch_bounds__(256) void gdn_conv_inputs_k4_kernel(GdnInArgs a, int CT) {
    constexpr int LPU = D / 8, UPB = 256 / LPU;
    const int U = 2 * a.HK + a.HV;
    const int ugroups = (U + UPB - 1) / UPB;
    const long n0 = (long)(blockIdx.x / ugroups) * CT;
    const int u = (blockIdx.x % ugroups) * UPB + (int)threadIdx.x / LPU;
    const int s = (int)threadIdx.x % LPU;
    const bool uv = u < U;                                // the unit exists (all lanes of a unit agree)
    const int uu = uv ? u : 0;
    const int kind = uu < a.HK ? 0 : (uu < 2 * a.HK ? 1 : 2);
    const int head = kind == 0 ? uu : (kind == 1 ? uu - a.HK : uu - 2 * a.HK);
    const long C = (long)U * D;
    const int c0 = (kind == 0 ? head * D : (kind == 1 ? (a.HK + head) * D : 2 * a.HK * D + head * D)) + 8 * s;
    const long n1 = n0 + CT < a.n_tok ? n0 + CT : a.n_tok;

    float w[4][8];                                        // w[j][e]: tap j (token n - j) of channel c0 + e
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const float4 wc = uv ? *reinterpret_cast<const float4*>(a.w + (long)(c0 + e) * 4) : make_float4(0.f, 0.f, 0.f, 0.f);
        w[0][e] = wc.w; w[1][e] = wc.z; w[2][e] = wc.y; w[3][e] = wc.x;
    }
    // sequence of n0
    int seq = 0, hi = a.num_seqs;
    while (hi - seq > 1) {
        const int mid = (seq + hi) >> 1;
        if (a.cu_seqlens[mid] <= n0) seq = mid;
        else hi = mid;
    }
    long seq0 = a.cu_seqlens[seq], seq_end = a.cu_seqlens[seq + 1];
    // rows n - 1, n - 2, n - 3 of the current token n
    float r1[8], r2[8], r3[8];
    auto fill = [&](long n) {
        load_tap<BF>(a, uv, n, 1, seq0, seq, C, c0, r1);
        load_tap<BF>(a, uv, n, 2, seq0, seq, C, c0, r2);
        load_tap<BF>(a, uv, n, 3, seq0, seq, C, c0, r3);
    };
    fill(n0);
    const int r = a.HV / a.HK;
    // gates of the block's tokens: lane s of a v unit takes tokens n0 + s, n0 + s + LPU, ..
    if (kind == 2 && uv) {
        const float dtb = a.dt_bias[head], ea = -__expf(a.A_log[head]);
        for (int i = s; i < CT; i += LPU) {
            const long n = n0 + i;
            if (n >= n1) break;
            const long gi = n * a.HV + head;
            const float xg = a.a[gi] + dtb;
            const float sp = xg > 20.f ? xg : log1pf(__expf(xg));
            a.g[gi] = ea * sp;
            a.beta[gi] = 1.f / (1.f + __expf(-a.b[gi]));
        }
    }
    for (long nb = n0; nb < n1; nb += CP) {
        float zr[CP][8];                                  // rows nb .. nb + CP - 1, loaded before the group's stores
#pragma unroll
        for (int i = 0; i < CP; ++i) load8<BF>(a.z, (nb + i) * a.z_st + c0, uv && nb + i < n1, zr[i]);
#pragma unroll
        for (int i = 0; i < CP; ++i) {
            const long n = nb + i;
            if (n >= n1) break;
            while (n == seq_end) {                        // a new sequence starts at n: rows before it from its prefix
                ++seq;
                seq0 = n;
                seq_end = a.cu_seqlens[seq + 1];
                fill(n);
            }
            float y[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float x = zr[i][e];
                y[e] = silu(w[0][e] * x + w[1][e] * r1[e] + w[2][e] * r2[e] + w[3][e] * r3[e]);
                r3[e] = r2[e];
                r2[e] = r1[e];
                r1[e] = x;
            }
            if (kind < 2) {
                float ss = 0.f;
#pragma unroll
                for (int e = 0; e < 8; ++e) ss += y[e] * y[e];
                ss = unit_sum<LPU>(ss);
                const float f = rsqrtf(ss + a.eps) * (kind == 0 ? a.q_scale : 1.f);
#pragma unroll
                for (int e = 0; e < 8; ++e) y[e] *= f;
                if (uv) {
                    void* dst = kind == 0 ? a.q : a.k;
                    for (int rr = 0; rr < r; ++rr) store8(dst, (n * a.HV + head * r + rr) * D + 8 * s, a.out_dtype, y);
                }
            } else if (uv) {
                store8(a.v, (n * a.HV + head) * D + 8 * s, a.out_dtype, y);
            }
        }
    }
}

template <int D, bool BF>
__global__ __launch_bounds__(256) void gated_norm_kernel(GatedNormArgs a) {
    constexpr int LPR = D / 8;
    const long tid = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long row = tid / LPR;
    const int s = (int)(tid % LPR);
    const bool valid = row < a.rows;
    const long e0 = (valid ? row : 0) * D + 8 * s;

    // BF: the layer runs in bf16 (gate and output bf16, the reference's bf16 rounding points); else all fp32
    float o[8], zg[8];
    if (a.o_dtype == DT_BF16) load8<true>(a.o, e0, valid, o);
    else load8<false>(a.o, e0, valid, o);
    if constexpr (BF) {
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = bf_round(o[e]);     // o.to(x.dtype)
    }
    load8<BF>(a.z, e0, valid, zg);
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) ss += o[e] * o[e];
    ss = unit_sum<LPR>(ss);
    const float inv = rsqrtf(ss / (float)D + a.eps);
    if (!valid) return;
    float r[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        if constexpr (BF) {
            const float h = bf_round(o[e] * inv);
            const float wh = bf_round(a.w[8 * s + e] * h);
            r[e] = wh * silu(zg[e]);
        } else {
            r[e] = a.w[8 * s + e] * (o[e] * inv) * silu(zg[e]);
        }
    }
    store8(a.out, e0, BF ? DT_BF16 : DT_F32, r);
}

// One token per sequence with a carried state, the whole layer between its projections in one launch: the conv over
// [prefix; z] with SiLU and l2norm, the gates, the delta-rule step, GatedNorm, and the new conv rows. Workgroup (h, b)
// holds value head h's whole state (D x D fp32, 16 rows of 4 columns per thread: D * D / 64 threads), so the row of o
// that the norm needs stays in the workgroup. Its loads go out before the small sums, which then cost no time of their
// own: the pass is bound by reading and writing the state once (134 MB at B = 32, HV = 32, D = 128). As separate
// kernels (conv pass, step, rounding, norm, the conv rows' concatenation and the parameters' casts to fp32, 15 launches
// of 2 .. 49 us) the same step took 140 us of GPU time and 260 us of the host's. With x, the gate logits (two products of
// 5120 x 32 by one row each, 11 us apiece as library calls) are formed here too, under the state's loads: the layer's step,
// its other projections included, went from 145 to
// 105 us at 32 sequences (d = 5120; D = 128. At D = 256 they would cost registers that the state needs).
__device__ __forceinline__ float ldp(const void* p, long i, int dt) {
    return dt == DT_BF16 ? bf2f(reinterpret_cast<const uint16_t*>(p)[i]) : reinterpret_cast<const float*>(p)[i];
}

template <int D, bool BF, bool XG>
__global__ __launch_bounds__(D * D / 64) void gdn_layer_step_kernel(GdnStepLayerArgs a) {
    constexpr int NT = D * D / 64, NW = NT / 64, CG = D / 4, RSTEP = NT / CG, RPT = D / RSTEP;
    static_assert(RPT == 16 && (CG == 16 || CG == 32 || CG == 64), "state split");
    __shared__ float qs[D], ks[D], vs[D], os[D];
    __shared__ __align__(16) float red[NW][D];
    __shared__ float sq[XG ? 4 : 2][NW];
    const int h = blockIdx.x, b = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int HK = a.HK, HV = a.HV, r = HV / HK, hk = h / r, K = a.K;
    const int cg = tid % CG, r0 = tid / CG;
    const long C = (long)(2 * HK + HV) * D, bh = (long)b * HV + h;
    using T = typename std::conditional<BF, uint16_t, float>::type;
    auto ld = [](const T* p) { if constexpr (BF) return bf2f(*p); else return *p; };
    float4 s[RPT];
#pragma unroll
    for (int i = 0; i < RPT; ++i) s[i] = nt_ldf4(a.s_in + (bh * D + r0 + RSTEP * i) * D + 4 * cg);

    // conv + SiLU of this head's q, k and v channels; the new conv rows (q and k by the first head that reads them)
    const T* z = reinterpret_cast<const T*>(a.z) + b * a.z_st;
    const T* pre = reinterpret_cast<const T*>(a.prefix) + (long)b * (K - 1) * C;
    T* nxt = reinterpret_cast<T*>(a.conv_out) + (long)b * (K - 1) * C;
    float ssq = 0.f, ssk = 0.f;
    for (int i = tid; i < 3 * D; i += NT) {
        const int kind = i / D, d = i % D;
        const long c = (kind == 0 ? hk : (kind == 1 ? HK + hk : 2 * HK + h)) * (long)D + d;
        const bool wr = kind == 2 || h % r == 0;
        const T z0 = z[c];
        float y = ld(&z0) * ldp(a.w, c * K + K - 1, a.w_dtype);
        if (wr) nxt[(K - 2) * C + c] = z0;
        for (int j = 1; j < K; ++j) {                    // the row j tokens back, weight column K - 1 - j
            const T x = a.prefix ? pre[(K - 1 - j) * C + c] : T(0);
            y = fmaf(ld(&x), ldp(a.w, c * K + K - 1 - j, a.w_dtype), y);
            if (wr && j < K - 1) nxt[(K - 2 - j) * C + c] = x;
        }
        y = silu(y);
        (kind == 0 ? qs : (kind == 1 ? ks : vs))[d] = y;
        if (kind == 0) ssq += y * y;
        else if (kind == 1) ssk += y * y;
    }
    // the gate logits of this head from the layer's input, 8 elements of x and of either weight row at a time
    float sa = 0.f, sb = 0.f;
    if constexpr (XG) {
        for (int i = 8 * tid; i < a.d; i += 8 * NT) {
            float xv[8], wa[8], wb[8];
            load8<BF>(a.x, b * a.x_st + i, true, xv);
            load8<BF>(a.a, (long)h * a.d + i, true, wa);
            load8<BF>(a.b, (long)h * a.d + i, true, wb);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                sa = fmaf(xv[e], wa[e], sa);
                sb = fmaf(xv[e], wb[e], sb);
            }
        }
    }
    ssq = unit_sum<64>(ssq);
    ssk = unit_sum<64>(ssk);
    if (lane == 0) { sq[0][wv] = ssq; sq[1][wv] = ssk; }
    if constexpr (XG) {
        sa = unit_sum<64>(sa);
        sb = unit_sum<64>(sb);
        if (lane == 0) { sq[2][wv] = sa; sq[3][wv] = sb; }
    }
    // gates, the same in every thread
    float al = 0.f, be = 0.f;
    auto gates = [&](float la, float lb) {
        const float ga = la + ldp(a.dt_bias, h, a.dt_dtype);
        const float gg = -__expf(ldp(a.A_log, h, a.al_dtype)) * (ga > 20.f ? ga : log1pf(__expf(ga)));
        al = __expf(gg);
        be = 1.f / (1.f + __expf(-lb));
    };
    if constexpr (!XG) gates(ldp(a.a, bh, a.io_dtype), ldp(a.b, bh, a.io_dtype));
    lds_barrier();
    float tq = 0.f, tk = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) { tq += sq[0][w]; tk += sq[1][w]; }
    if constexpr (XG) {                                  // (rounded as the projections' outputs are)
        float la = 0.f, lb = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) { la += sq[2][w]; lb += sq[3][w]; }
        gates(BF ? bf_round(la) : la, BF ? bf_round(lb) : lb);
    }
    const float fq = rsqrtf(tq + a.l2_eps) * a.q_scale, fk = rsqrtf(tk + a.l2_eps);

    // sum over the rows: lanes of one column group in the wave, then the waves
    auto col_sum = [&](const float* x, float f, float (&out)[4]) {
        float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < RPT; ++i) {
            const float xr = x[r0 + RSTEP * i] * f;
            v[0] += xr * s[i].x; v[1] += xr * s[i].y; v[2] += xr * s[i].z; v[3] += xr * s[i].w;
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
#pragma unroll
            for (int off = CG; off < 64; off <<= 1) v[e] += __shfl_xor(v[e], off);
        }
        if constexpr (NW > 1) {
            if (lane < CG) *reinterpret_cast<float4*>(&red[wv][4 * cg]) = make_float4(v[0], v[1], v[2], v[3]);
            lds_barrier();
#pragma unroll
            for (int e = 0; e < 4; ++e) out[e] = 0.f;
#pragma unroll
            for (int w = 0; w < NW; ++w) {
                const float4 p = *reinterpret_cast<const float4*>(&red[w][4 * cg]);
                out[0] += p.x; out[1] += p.y; out[2] += p.z; out[3] += p.w;
            }
            lds_barrier();
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) out[e] = v[e];
        }
    };
    float rc[4], dl[4], o4[4];
    col_sum(ks, fk, rc);
#pragma unroll
    for (int e = 0; e < 4; ++e) dl[e] = be * (vs[4 * cg + e] - al * rc[e]);
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
        const float k = ks[r0 + RSTEP * i] * fk;
        s[i].x = al * s[i].x + k * dl[0];
        s[i].y = al * s[i].y + k * dl[1];
        s[i].z = al * s[i].z + k * dl[2];
        s[i].w = al * s[i].w + k * dl[3];
        nt_stf4(a.s_out + (bh * D + r0 + RSTEP * i) * D + 4 * cg, s[i]);
    }
    col_sum(qs, fq, o4);
    if (r0 == 0) {
#pragma unroll
        for (int e = 0; e < 4; ++e) os[4 * cg + e] = BF ? bf_round(o4[e]) : o4[e];    // o.to(x.dtype)
    }
    lds_barrier();
    // GatedNorm of the head's row by the first D / 8 lanes, as gated_norm_kernel
    constexpr int LPR = D / 8;
    if (tid < LPR) {
        float o[8], zg[8], out[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = os[8 * tid + e];
        load8<BF>(a.zg, bh * D + 8 * tid, true, zg);
        float ss = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) ss += o[e] * o[e];
        ss = unit_sum<LPR>(ss);
        const float inv = rsqrtf(ss / (float)D + a.eps);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float w = ldp(a.norm_w, 8 * tid + e, a.nw_dtype);
            if constexpr (BF) out[e] = bf_round(w * bf_round(o[e] * inv)) * silu(zg[e]);
            else out[e] = w * (o[e] * inv) * silu(zg[e]);
        }
        store8(a.out, bh * D + 8 * tid, BF ? DT_BF16 : DT_F32, out);
    }
}

int gdn_layer_step_dispatch(const GdnStepLayerArgs& a, hipStream_t stream) {
    const dim3 grid((unsigned)a.HV, (unsigned)a.B), block((unsigned)(a.D * a.D / 64));
    const bool bf = a.io_dtype == DT_BF16;
    auto go = [&](auto k16, auto k32) {
        if (bf) hipLaunchKernelGGL(k16, grid, block, 0, stream, a);
        else hipLaunchKernelGGL(k32, grid, block, 0, stream, a);
    };
    switch (a.D) {
        case 64: if (a.x) go(gdn_layer_step_kernel<64, true, true>, gdn_layer_step_kernel<64, false, true>);
                 else go(gdn_layer_step_kernel<64, true, false>, gdn_layer_step_kernel<64, false, false>); break;
        case 128: if (a.x) go(gdn_layer_step_kernel<128, true, true>, gdn_layer_step_kernel<128, false, true>);
                  else go(gdn_layer_step_kernel<128, true, false>, gdn_layer_step_kernel<128, false, false>); break;
        case 256: if (a.x) return BF_ERR_UNSUPPORTED;
                  go(gdn_layer_step_kernel<256, true, false>, gdn_layer_step_kernel<256, false, false>); break;
        default: return BF_ERR_UNSUPPORTED;
    }
    return (int)hipGetLastError();
}

int gdn_conv_inputs_dispatch(const GdnInArgs& a, hipStream_t stream) {
    const long threads = a.n_tok * (2 * a.HK + a.HV) * (a.D / 8);
    if (threads == 0) return 0;
    if (a.K == 4) {
        const int upb = 256 / (a.D / 8), U = 2 * a.HK + a.HV;
        const int ug = (U + upb - 1) / upb, ct = conv_block(a.n_tok, ug);
        const long blocks = ((a.n_tok + ct - 1) / ct) * ug;
        if (blocks > 0x7fffffffL) return BF_STATUS_INVALID;
        const dim3 grid((unsigned)blocks), block(256);
        const bool bf = a.in_dtype == DT_BF16;
        switch (a.D) {
            case 64: if (bf) hipLaunchKernelGGL((gdn_conv_inputs_k4_kernel<64, true>), grid, block, 0, stream, a, ct);
                     else hipLaunchKernelGGL((gdn_conv_inputs_k4_kernel<64, false>), grid, block, 0, stream, a, ct); break;
            case 128: if (bf) hipLaunchKernelGGL((gdn_conv_inputs_k4_kernel<128, true>), grid, block, 0, stream, a, ct);
                      else hipLaunchKernelGGL((gdn_conv_inputs_k4_kernel<128, false>), grid, block, 0, stream, a, ct); break;
            case 256: if (bf) hipLaunchKernelGGL((gdn_conv_inputs_k4_kernel<256, true>), grid, block, 0, stream, a, ct);
                      else hipLaunchKernelGGL((gdn_conv_inputs_k4_kernel<256, false>), grid, block, 0, stream, a, ct); break;
            default: return BF_ERR_UNSUPPORTED;
        }
        return (int)hipGetLastError();
    }
    const long blocks = (threads + 255) / 256;
    if (blocks > 0x7fffffffL) return BF_STATUS_INVALID;
    const dim3 grid((unsigned)blocks), block(256);
    auto launch = [&](bool b16, auto kb, auto kf) {
        if (b16) hipLaunchKernelGGL(kb, grid, block, 0, stream, a);
        else hipLaunchKernelGGL(kf, grid, block, 0, stream, a);
    };
    const bool bf = a.in_dtype == DT_BF16;
    switch (a.D) {
        case 64: launch(bf, gdn_conv_inputs_kernel<64, true>, gdn_conv_inputs_kernel<64, false>); break;
        case 128: launch(bf, gdn_conv_inputs_kernel<128, true>, gdn_conv_inputs_kernel<128, false>); break;
        case 256: launch(bf, gdn_conv_inputs_kernel<256, true>, gdn_conv_inputs_kernel<256, false>); break;
        default: return BF_ERR_UNSUPPORTED;
    }
    return (int)hipGetLastError();
}

int gated_norm_dispatch(const GatedNormArgs& a, hipStream_t stream) {
    const long threads = a.rows * (a.D / 8);
    if (threads == 0) return 0;
    const long blocks = (threads + 255) / 256;
    if (blocks > 0x7fffffffL) return BF_STATUS_INVALID;
    const dim3 grid((unsigned)blocks), block(256);
    auto launch = [&](bool b16, auto kb, auto kf) {
        if (b16) hipLaunchKernelGGL(kb, grid, block, 0, stream, a);
        else hipLaunchKernelGGL(kf, grid, block, 0, stream, a);
    };
    const bool bf = a.io_dtype == DT_BF16;
    switch (a.D) {
        case 64: launch(bf, gated_norm_kernel<64, true>, gated_norm_kernel<64, false>); break;
        case 128: launch(bf, gated_norm_kernel<128, true>, gated_norm_kernel<128, false>); break;
        case 256: launch(bf, gated_norm_kernel<256, true>, gated_norm_kernel<256, false>); break;
        default: return BF_ERR_UNSUPPORTED;
    }
    return (int)hipGetLastError();
}

}  // namespace bf
