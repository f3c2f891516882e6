// K2, fp32 operands: exact sliding-window + sink attention over a prefill chunk, with per-row log-sum-exp and the fused
// gamma mix.
//
// Reference: HybridAttention._window_fp32 (Heimdall/heimdall/hibrit.py:341-361) and the mix of :409-411.
// Query i of the chunk sits at absolute position p = start + i. Visible keys (mask of hibrit.py:356):
//   sinks j < n_sinks with j <= p, and window keys at positions kp with S <= kp <= p, p - kp < W, where
//   kp < start comes from the ring (slot kp mod W, valid iff ring_pos[slot] == kp) and kp >= start from the chunk.
// s = (q . k) / sqrt(D); lse = ln sum_visible e^s; o_win = softmax(s) V.
// Mix (when enabled): gamma = sigmoid(z + mix_lse (lse - ln W)) [p >= W]; o = o_win + gamma (mem_scale o_mem - o_win).
//
// Bound by the matrix cores: both products run on bf16 MFMAs over three exact bf16 planes per fp32 operand (Planes,
// bf_common.h), 0.375 of the cycles of the fp32 MFMA. One workgroup = NW waves x 16 queries of one query head, Q's
// planes in registers. Keys come in blocks of 32: their K and V rows are loaded as fp32 and stored to LDS as planes,
// K_{i+1} while V_i is multiplied and V_i while K_i is, so each needs one tile and the loads are in flight for half a
// block. Of the two waves of a SIMD (NW = 8) one stores its share before its products and the other after them, so the
// VALU work of one runs beside the MFMAs of the other. Scores are computed transposed (S^T = K Q^T) so each lane's
// softmax statistics belong to its own query column, and P feeds the P V product straight from registers.
// 4096 tokens, H = 16, G = 4, D = 256, W = 2048 + 4: 1810 -> 905 us (kernel alone).
#include "bf_common.h"
#include "bf_internal.h"

namespace bf {

constexpr int W32_KB = 32;       // keys per block

template <int D>
struct W32Shared {
    // rows padded by 16 and 32 bytes: the 16 rows of a K fragment read, and the 4-row pieces of a transposing V read,
    // fall into distinct banks
    uint16_t k[3][W32_KB][D + 8];
    uint16_t v[3][W32_KB][D + 16];
    int krel[W32_KB];            // key position minus the workgroup's first query position; INT_MAX: not a key
};

// The keys of a workgroup are split into segments that each come from one contiguous source: the sinks, the ring
// up to its wrap point, the ring after it, and the chunk. A key block never straddles two segments, so the address
// of every row is base + min(row, last) * stride with no per-row branching.
struct KeySeg {
    const float* kb;   // first key row of the segment
    const float* vb;   // first value row
    long ks, vs;       // row strides (elements)
    long pos0;         // position of the first row (sinks: 0)
    int count;         // rows
    int slot0;         // ring slot of the first row, or -1 outside the ring
    int sink;          // sink rows: visible to every query at or after their position, no window limit
};

// A thread's share of a key or value block: NCH pieces of 8 consecutive elements, of rows past the segment's end its
// last row again (their scores are masked; exec-masked loads would make the compiler wait for the whole prefetch early).
template <int D, int NT>
struct W32Rows {
    static constexpr int CPR = D / 8, N = W32_KB * CPR, NCH = (N + NT - 1) / NT;
    float4 x[NCH][2];
    __device__ __forceinline__ void load(const float* base, long stride, int last) {
#pragma unroll
        for (int j = 0; j < NCH; ++j) {
            const int c = threadIdx.x + NT * j;
            if (N % NT == 0 || c < N) {
                const float* p = base + min(c / CPR, last) * stride + 8 * (c % CPR);
                x[j][0] = *reinterpret_cast<const float4*>(p);
                x[j][1] = *reinterpret_cast<const float4*>(p + 4);
            }
        }
    }
    template <int P>
    __device__ __forceinline__ void park(uint16_t (&t)[3][W32_KB][P]) const {
#pragma unroll
        for (int j = 0; j < NCH; ++j) {
            const int c = threadIdx.x + NT * j;
            if (N % NT == 0 || c < N) {
                const Planes s = split8(x[j][0], x[j][1]);
#pragma unroll
                for (int i = 0; i < 3; ++i) st16(&t[i][c / CPR][8 * (c % CPR)], s.p[i]);
            }
        }
    }
};

template <int D, int NW, bool BO>
__global__ __launch_bounds__(64 * NW) void window_kernel(WinArgs a) {
    constexpr int KB = W32_KB, NT = 64 * NW, BQ = 16 * NW;
    constexpr int NKD = D / 32;           // fragments along D
    constexpr int NDT = D / 16;           // d tiles of the output
    __shared__ W32Shared<D> sm;

    // items of one KV head on neighbouring dispatch slots of an XCD, the ones with most keys first (WinMap)
    const int R = a.R, G = a.G, H = G * R, nqb = (a.T + BQ - 1) / BQ;
    const long wi = window_item(a.map, (int)(blockIdx.x % 8), blockIdx.x / 8);
    if (wi < 0) return;
    const int r = (int)(wi % R);
    long rest = wi / R;
    const int qb = nqb - 1 - (int)(rest % nqb);
    rest /= nqb;
    const int g = (int)(rest % G), b = (int)(rest / G), h = g * R + r;
    const int lane = lane_id(), wv = wave_id(), l16 = lane & 15, lg = lane >> 4;
    const long qi0 = (long)qb * BQ;                       // first query index of the workgroup
    const int nq = (int)min((long)BQ, (long)a.T - qi0);
    const long p_first = a.start + qi0, p_last = a.start + qi0 + nq - 1;
    const float scale = rsqrtf((float)D);

    const float* Qb = reinterpret_cast<const float*>(a.q) + b * a.q_sb + h * a.q_sh;
    const float* rk = a.ring_k ? reinterpret_cast<const float*>(a.ring_k) + ((long)b * G + g) * a.W * D : nullptr;
    const float* rv = a.ring_v ? reinterpret_cast<const float*>(a.ring_v) + ((long)b * G + g) * a.W * D : nullptr;
    const float* ck = reinterpret_cast<const float*>(a.k) + b * a.k_sb + g * a.k_sh;
    const float* cv = reinterpret_cast<const float*>(a.v) + b * a.v_sb + g * a.v_sh;
    const float* sk = a.n_sinks ? reinterpret_cast<const float*>(a.sink_k) + ((long)b * G + g) * a.n_sinks * D : nullptr;
    const float* sv = a.n_sinks ? reinterpret_cast<const float*>(a.sink_v) + ((long)b * G + g) * a.n_sinks * D : nullptr;

    // Q planes (B operand of S^T = K Q^T): column l16, k range 8 lg of each 32-wide step
    const int qrel = 16 * wv + l16;                       // query position minus p_first
    Planes fq[NKD];
    {
        const float* qrow = Qb + (qi0 + min(qrel, nq - 1)) * a.q_st;
#pragma unroll
        for (int kf = 0; kf < NKD; ++kf)
            fq[kf] = split8(*reinterpret_cast<const float4*>(qrow + 32 * kf + 8 * lg),
                            *reinterpret_cast<const float4*>(qrow + 32 * kf + 8 * lg + 4));
    }
    f32x4 o[NDT];
    float m = -INFINITY, l = 0.f;
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};

    // key segments (sinks, ring before its wrap point, ring after it, chunk), consumed in blocks of KB rows
    const long kp_lo = max((long)a.sinks, p_first - a.W + 1);
    KeySeg sg[4];
    int nb[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        sg[j] = KeySeg{ck, cv, 0, 0, 0, 0, -1, 0};
        nb[j] = 0;
    }
    if (a.n_sinks) sg[0] = KeySeg{sk, sv, D, D, 0, a.n_sinks, -1, 1};
    const long rhi = min(p_last, a.start - 1);
    if (rk && kp_lo <= rhi) {
        const int sa = (int)(kp_lo % a.W);                  // one division per workgroup
        const long n = rhi - kp_lo + 1;
        const long n1 = min(n, (long)(a.W - sa));
        sg[1] = KeySeg{rk + (long)sa * D, rv + (long)sa * D, D, D, kp_lo, (int)n1, sa, 0};
        if (n > n1) sg[2] = KeySeg{rk, rv, D, D, kp_lo + n1, (int)(n - n1), 0, 0};
    }
    const long clo = max(kp_lo, a.start);
    if (clo <= p_last)
        sg[3] = KeySeg{ck + (clo - a.start) * a.k_st, cv + (clo - a.start) * a.v_st, a.k_st, a.v_st, clo,
                       (int)(p_last - clo + 1), -1, 0};
    int nblk = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        nb[j] = (sg[j].count + KB - 1) / KB;
        nblk += nb[j];
    }
    // block i as a segment of its own: the KB rows starting at row KB * (i - first block of its segment)
    auto block_ref = [&](int i) {
        KeySeg s = sg[3];
        int base = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (i >= base && i < base + nb[j]) {
                const int off = (i - base) * KB;
                s = sg[j];
                s.kb += off * sg[j].ks;
                s.vb += off * sg[j].vs;
                s.pos0 += off;
                s.count -= off;
                if (s.slot0 >= 0) s.slot0 += off;
            }
            base += nb[j];
        }
        return s;
    };

    const rsrc_t rpos = make_rsrc(a.ring_pos, a.ring_pos ? (uint32_t)a.W * 8u : 0u);
    W32Rows<D, NT> kr, vr;
    uint2 rp;                                             // ring_pos of row (thread % KB) of a ring block
    KeySeg br, nx;                                        // this block and the next
    auto fetch_k = [&](const KeySeg& s) {
        const int last = min(s.count, KB) - 1;
        // out-of-range offset (outside the ring) reads 0
        rp = buf_ld8(rpos, s.slot0 >= 0 ? (uint32_t)(s.slot0 + min((int)threadIdx.x % KB, last)) * 8u : 0xFFFFFFF0u);
        kr.load(s.kb, s.ks, last);
    };
    auto park_k = [&](const KeySeg& s) {
        kr.park(sm.k);
        if (threadIdx.x < KB) {
            const long kp = s.pos0 + threadIdx.x;
            bool val = (int)threadIdx.x < s.count;
            if (s.slot0 >= 0) val = val && (long)(((uint64_t)rp.y << 32) | rp.x) == kp;
            // sinks far behind the chunk clamp (always visible)
            sm.krel[threadIdx.x] = val ? (int)max(kp - p_first, -(1L << 30)) : 0x7fffffff;
        }
    };
    if (nblk > 0) {
        br = block_ref(0);
        fetch_k(br);
        vr.load(br.vb, br.vs, min(br.count, KB) - 1);
        park_k(br);
    }
    const bool early = NW < 8 || wv < NW / 2;             // this wave stores its share before its products
    const int trow = 4 * lg + (l16 >> 2), tcol = 4 * (l16 & 3);
    for (int i = 0; i < nblk; ++i) {
        const bool more = i + 1 < nblk;
        __syncthreads();                                   // K_i is in LDS, V_{i-1} fully consumed
        if (more) {
            nx = block_ref(i + 1);
            fetch_k(nx);
        }
        // the wave's queries see something of the block: its first key is not past them all, its last one not behind
        // all of their windows
        const long k0 = br.pos0 - p_first, k1 = k0 + min(br.count, KB) - 1;
        const bool on = 16 * wv < nq && k0 <= 16 * wv + 15 && (br.sink || 16 * wv - k1 < a.W);
        if (early) vr.park(sm.v);
        f32x4 s[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
        float corr = 1.f;
        if (on) {
            // S^T = K Q^T for this block
#pragma unroll
            for (int kf = 0; kf < NKD; ++kf)
#pragma unroll
                for (int kt = 0; kt < 2; ++kt) {
                    Planes ak;
#pragma unroll
                    for (int j = 0; j < 3; ++j) ak.p[j] = ld16(&sm.k[j][16 * kt + l16][32 * kf + 8 * lg]);
                    mma3(s[kt], ak, fq[kf]);
                }
            // mask, online softmax per query column
            float bm = -INFINITY;
#pragma unroll
            for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int kp = sm.krel[16 * kt + 4 * lg + e];
                    const bool vis = kp <= qrel && (br.sink || qrel - kp < a.W);
                    const float x = vis ? s[kt][e] * scale : -INFINITY;
                    s[kt][e] = x;
                    bm = fmaxf(bm, x);
                }
            bm = fmaxf(bm, __shfl_xor(bm, 16));
            bm = fmaxf(bm, __shfl_xor(bm, 32));
            const float mn = fmaxf(m, bm);
            corr = mn == -INFINITY ? 1.f : __expf(m - mn);
            float ls = 0.f;
#pragma unroll
            for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float p = mn == -INFINITY ? 0.f : __expf(s[kt][e] - mn);
                    s[kt][e] = p;
                    ls += p;
                }
            ls += __shfl_xor(ls, 16);
            ls += __shfl_xor(ls, 32);
            l = l * corr + ls;
            m = mn;
        }
        if (!early) vr.park(sm.v);
        __syncthreads();                                   // V_i is in LDS, K_i fully consumed
        if (more) {
            vr.load(nx.vb, nx.vs, min(nx.count, KB) - 1);
            if (early) park_k(nx);
        }
        if (on) {
            if (__any(corr != 1.f)) {
#pragma unroll
                for (int dt = 0; dt < NDT; ++dt) {
                    o[dt][0] *= corr; o[dt][1] *= corr; o[dt][2] *= corr; o[dt][3] *= corr;
                }
            }
            // O^T += V^T P^T: the K index 8 lg + e is key 4 lg + e of the first 16 (e < 4) or of the second
            const Planes pb = split8(make_float4(s[0][0], s[0][1], s[0][2], s[0][3]),
                                     make_float4(s[1][0], s[1][1], s[1][2], s[1][3]));
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt) {
                Planes av;
#pragma unroll
                for (int j = 0; j < 3; ++j) {
                    const uint2 lo = lds_tr16(reinterpret_cast<const char*>(&sm.v[j][trow][16 * dt + tcol]));
                    const uint2 hi = lds_tr16(reinterpret_cast<const char*>(&sm.v[j][16 + trow][16 * dt + tcol]));
                    av.p[j] = make_uint4(lo.x, lo.y, hi.x, hi.y);
                }
                mma3(o[dt], av, pb);
            }
        }
        if (more && !early) park_k(nx);
        br = nx;
    }

    // epilogue: normalise, lse, gamma mix, store o [B][T][H][D]
    const int qi = qrel;
    if (qi >= nq) return;
    const float lnW = logf((float)a.W);
    const long tq = qi0 + qi;
    const float inv = 1.f / l;
    const float lse = m + logf(l);
    if (a.lse && lg == 0) a.lse[((long)b * H + h) * a.T + tq] = lse;
    float gam = 0.f;
    if (a.mix_on && p_first + qrel >= a.W)
        gam = 1.f / (1.f + __expf(-(a.z[((long)b * a.T + tq) * H + h] + a.mix_lse[h] * (lse - lnW))));
    const float ms = a.mix_on ? a.mem_scale[h] : 0.f;
    const long orow = (((long)b * a.T + tq) * H + h) * D;
    // memory reads issued together (every row of o_mem exists); rows with gam = 0 keep the window output by
    // selection, so rows the delta rule never wrote cannot leak in
    const bool mixed = gam != 0.f;
    float4 om[NDT];
    if (a.mix_on) load_om<NDT>(a, orow + 4 * lg, om);
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) {
        const int d0 = 16 * dt + 4 * lg;
        float r4[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) r4[e] = o[dt][e] * inv;
        if (a.mix_on) {
            const float mv[4] = {om[dt].x, om[dt].y, om[dt].z, om[dt].w};
#pragma unroll
            for (int e = 0; e < 4; ++e) r4[e] = mixed ? r4[e] + gam * (ms * mv[e] - r4[e]) : r4[e];
        }
        if constexpr (BO) store4<BF16>(reinterpret_cast<uint16_t*>(a.o) + orow + d0, r4[0], r4[1], r4[2], r4[3]);
        else store4<F32>(reinterpret_cast<float*>(a.o) + orow + d0, r4[0], r4[1], r4[2], r4[3]);
    }
}

template <int D, int NW>
static int launch_window(const WinArgs& args, hipStream_t stream) {
    WinArgs a = args;
    // the map counts 128-query items; 64-query ones are those of twice the length
    const int f = a.start < a.W ? 2 : 1;
    a.map = window_map_make(a.B, a.G, a.R, a.T * (8 / NW), f, 0);
    if (8 * a.map.per > 0x7fffffffL || a.T > (1 << 30)) return BF_STATUS_INVALID;
    const dim3 grid((unsigned)(8 * a.map.per)), block(64 * NW);
    if (a.o_dtype == DT_BF16) hipLaunchKernelGGL((window_kernel<D, NW, true>), grid, block, 0, stream, a);
    else hipLaunchKernelGGL((window_kernel<D, NW, false>), grid, block, 0, stream, a);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : (int)e;
}

// 64 queries per workgroup while that leaves every workgroup a CU of its own (half the waves per SIMD share the same
// chain of blocks); above, 128, which store each key block to LDS half as often.
template <int D>
static int launch_window_by_size(const WinArgs& a, hipStream_t stream) {
    const bool few = (long)a.B * a.G * a.R * ((a.T + 63L) / 64) <= 256;
    return few ? launch_window<D, 4>(a, stream) : launch_window<D, 8>(a, stream);
}

int window_dispatch(const WinArgs& a, hipStream_t stream) {
    if (a.in_dtype == DT_BF16) return window_fa_dispatch(a, stream);
    switch (a.D) {
        case 64: return launch_window_by_size<64>(a, stream);
        case 128: return launch_window_by_size<128>(a, stream);
        case 256: return launch_window_by_size<256>(a, stream);
        default: return BF_ERR_UNSUPPORTED;
    }
}

}  // namespace bf
