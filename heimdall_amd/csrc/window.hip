// K2, fp32 operands: exact sliding-window + sink attention over a prefill chunk, with per-row log-sum-exp and the fused
// gamma mix.
//
// (D = 64 over few queries or a short window: window_d64.hip.)
// Reference: HybridAttention._window_fp32 (Heimdall/heimdall/hibrit.py:341-361) and the mix of :409-411.
// Query i of the chunk sits at absolute position p = start + i. Visible keys (mask of hibrit.py:356):
//   sinks j < n_sinks with j <= p, and window keys at positions kp with S <= kp <= p, p - kp < W, where
//   kp < start comes from the ring (slot kp mod W, valid iff ring_pos[slot] == kp) and kp >= start from the chunk.
// s = (q . k) / sqrt(D); lse = ln sum_visible e^s; o_win = softmax(s) V.
// Mix (when enabled): gamma = sigmoid(z + mix_lse (lse - ln W)) [p >= W]; o = o_win + gamma (mem_scale o_mem - o_win).
//
// Both products run on bf16 MFMAs over three exact bf16 planes per fp32 operand (Planes, bf_common.h), 0.375 of the cycles
// of the fp32 MFMA. One workgroup = NW / 2 pairs of waves, a pair 32 queries of one query head: each wave holds the planes
// of one half of the queries' dims and that half of the output, so a fragment read from LDS feeds twelve MFMAs within half
// the registers (16 queries and all dims per wave read twice the bytes, as many cycles of LDS as of MFMA: 790 us in the
// case below; 32 queries and all dims spill). The pair adds its two partial scores through LDS. Keys come in blocks of 32:
// their K and V rows are loaded as fp32 and stored to LDS as planes, K_{i+1} between the MFMAs of V_i and V_i between
// those of K_i, so each needs one tile, two barriers a block and half the registers: a piece of K is loaded where one of V was stored. Scores are
// computed transposed (S^T = K Q^T) so each lane's softmax statistics belong to its own query column, and P feeds the P V
// product straight from registers.
// 4096 tokens, H = 16, G = 4, D = 256, W = 2048 + 4: 1765 us with fp32 MFMAs, now 785 us (window kernel alone; 750 with a split
// that cut the first plane off and made infinities NaN).
#include "bf_common.h"
#include "bf_internal.h"

namespace bf {

constexpr int W32_KB = 32;       // keys per block

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
// The same value in every lane: moved to scalar registers.
__device__ __forceinline__ long uniform(long x) {
    return (long)(((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(x >> 32)) << 32) |
                  (uint32_t)__builtin_amdgcn_readfirstlane((int)x));
}
__device__ __forceinline__ KeySeg uniform(const KeySeg& s) {
    return KeySeg{reinterpret_cast<const float*>(uniform(reinterpret_cast<long>(s.kb))),
                  reinterpret_cast<const float*>(uniform(reinterpret_cast<long>(s.vb))), uniform(s.ks), uniform(s.vs),
                  uniform(s.pos0), __builtin_amdgcn_readfirstlane(s.count), __builtin_amdgcn_readfirstlane(s.slot0),
                  __builtin_amdgcn_readfirstlane(s.sink)};
}

template <int D, int NW>
struct W32Shared {
    // rows padded by 16 and 32 bytes: the 16 rows of a K fragment read, and the 4-row pieces of a transposing V read,
    // fall into distinct banks
    uint16_t k[3][W32_KB][D + 8];
    uint16_t v[3][W32_KB][D + 16];
    __align__(16) int krel[2][W32_KB];   // by block parity: key position minus the workgroup's first query position; INT_MAX: not a key
    int nval[2];                         // by block parity: its keys
    KeySeg seg[4];
    f32x4 part[NW][4][64];       // partial scores of each wave: [query tile x key tile][lane]
};

// A thread's share of a key or value block: pieces of 4 consecutive elements, a wave's instruction taking 256 / D whole
// rows (at D = 256 a row's address is scalar). Rows past the segment's end are its last row again (their scores are
// masked; exec-masked loads would make the compiler wait for the whole prefetch early).
template <int D, int NW>
struct W32Rows {
    static constexpr int RPL = 256 / D, NCH = W32_KB / (RPL * NW);
    static_assert(NCH * RPL * NW == W32_KB, "rows of a block");
    f32x4 x[NCH];
    __device__ __forceinline__ static int row(int wv, int lane, int j) { return (wv + NW * j) * RPL + (RPL > 1 ? lane / (D / 4) : 0); }
    __device__ __forceinline__ void load(const float* kv, long stride, int last, int wv, int lane, int j) {
        // (a base that came through LDS is a generic pointer to the compiler: say that it is global memory)
        typedef __attribute__((address_space(1))) const f32x4 gf4;
        typedef __attribute__((address_space(1))) const float gf;
        gf* rp = (gf*)kv + min(row(wv, lane, j), last) * stride;
        x[j] = *reinterpret_cast<gf4*>(rp + 4 * (lane % (D / 4)));
    }
    template <int P>
    __device__ __forceinline__ void park(uint16_t (&t)[3][W32_KB][P], int wv, int lane, int j) {
        uint2 s[3];
        // opaque here, or the split moves up out of the two branches that store the piece, into more registers
        asm volatile("" : "+v"(x[j]));
        split_pair<SPLIT_ANY>(x[j][0], x[j][1], s[0].x, s[1].x, s[2].x);
        split_pair<SPLIT_ANY>(x[j][2], x[j][3], s[0].y, s[1].y, s[2].y);
#pragma unroll
        for (int i = 0; i < 3; ++i) *reinterpret_cast<uint2*>(&t[i][row(wv, lane, j)][4 * (lane % (D / 4))]) = s[i];
    }
};

template <int D, int NW, bool BO>
__global__ __launch_bounds__(64 * NW) void window_kernel(WinArgs a) {
    constexpr int KB = W32_KB, QT = 2, QW = 16 * QT, BQ = QW * NW / 2;
    constexpr int NKD = D / 64;           // fragments along a wave's half of D
    constexpr int NDT = D / 32;           // d tiles of its half of the output
    __shared__ W32Shared<D, NW> sm;

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
    const int pr = wv % (NW / 2), dh = wv / (NW / 2) * (D / 2), mate = wv ^ (NW / 2);   // pair, first dim, the other wave
    const long qi0 = (long)qb * BQ;                       // first query index of the workgroup
    const int nq = (int)min((long)BQ, (long)a.T - qi0);
    const long p_first = a.start + qi0, p_last = a.start + qi0 + nq - 1;
    const float scale = rsqrtf((float)D), scale2 = scale * 1.4426950408889634f;

    const float* Qb = reinterpret_cast<const float*>(a.q) + b * a.q_sb + h * a.q_sh;
    const float* rk = a.ring_k ? reinterpret_cast<const float*>(a.ring_k) + ((long)b * G + g) * a.W * D : nullptr;
    const float* rv = a.ring_v ? reinterpret_cast<const float*>(a.ring_v) + ((long)b * G + g) * a.W * D : nullptr;
    const float* ck = reinterpret_cast<const float*>(a.k) + b * a.k_sb + g * a.k_sh;
    const float* cv = reinterpret_cast<const float*>(a.v) + b * a.v_sb + g * a.v_sh;
    const float* sk = a.n_sinks ? reinterpret_cast<const float*>(a.sink_k) + ((long)b * G + g) * a.n_sinks * D : nullptr;
    const float* sv = a.n_sinks ? reinterpret_cast<const float*>(a.sink_v) + ((long)b * G + g) * a.n_sinks * D : nullptr;

    // Q planes (B operand of S^T = K Q^T): column l16, k range 8 lg of each 32-wide step
    const int qrel = QW * pr + l16;                       // tile 0's query position minus p_first (tile qt: + 16 qt)
    Planes fq[QT][NKD];
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
        const float* qrow = Qb + (qi0 + min(qrel + 16 * qt, nq - 1)) * a.q_st + dh;
#pragma unroll
        for (int kf = 0; kf < NKD; ++kf)
            fq[qt][kf] = split8<SPLIT_ANY>(*reinterpret_cast<const f32x4*>(qrow + 32 * kf + 8 * lg),
                                           *reinterpret_cast<const f32x4*>(qrow + 32 * kf + 8 * lg + 4));
    }
    f32x4 o[QT][NDT];
    float m[QT], l[QT];
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
        m[qt] = -INFINITY;
        l[qt] = 0.f;
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) o[qt][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    }

    // key segments (sinks, ring before its wrap point, ring after it, chunk), consumed in blocks of KB rows; they are kept
    // in LDS, since four of them do not fit the scalar registers beside the loop's
    const long kp_lo = max((long)a.sinks, p_first - a.W + 1);
    const long rhi = min(p_last, a.start - 1), clo = max(kp_lo, a.start);
    const int sa = rk && kp_lo <= rhi ? (int)(kp_lo % a.W) : 0;              // one division per workgroup
    const long nr = rk && kp_lo <= rhi ? rhi - kp_lo + 1 : 0, n1 = min(nr, (long)(a.W - sa));
    const int cnt[4] = {a.n_sinks, (int)n1, (int)(nr - n1), clo <= p_last ? (int)(p_last - clo + 1) : 0};
    int end[4];                                            // first block past each segment
#pragma unroll
    for (int j = 0; j < 4; ++j) end[j] = (j ? end[j - 1] : 0) + (cnt[j] + KB - 1) / KB;
    const int nblk = end[3];
    if (threadIdx.x == 0) {
        sm.seg[0] = KeySeg{sk, sv, D, D, 0, cnt[0], -1, 1};
        sm.seg[1] = KeySeg{rk + (long)sa * D, rv + (long)sa * D, D, D, kp_lo, cnt[1], sa, 0};
        sm.seg[2] = KeySeg{rk, rv, D, D, kp_lo + n1, cnt[2], 0, 0};
        sm.seg[3] = KeySeg{ck + (clo - a.start) * a.k_st, cv + (clo - a.start) * a.v_st, a.k_st, a.v_st, clo, cnt[3], -1, 0};
    }
    __syncthreads();
    // block i as a segment of its own: the KB rows starting at row KB * (i - first block of its segment)
    auto block_ref = [&](int i) {
        const int j = i < end[0] ? 0 : i < end[1] ? 1 : i < end[2] ? 2 : 3;
        const int off = (i - (j == 0 ? 0 : j == 1 ? end[0] : j == 2 ? end[1] : end[2])) * KB;
        KeySeg s = uniform(sm.seg[j]);
        s.kb += off * s.ks;
        s.vb += off * s.vs;
        s.pos0 += off;
        s.count -= off;
        if (s.slot0 >= 0) s.slot0 += off;
        return s;
    };

    const rsrc_t rpos = make_rsrc(a.ring_pos, a.ring_pos ? (uint32_t)a.W * 8u : 0u);
    constexpr int NCH = W32Rows<D, NW>::NCH, NP = NCH / NKD;   // pieces per step
    static_assert(NCH == NP * NKD && 2 * NKD == NDT, "pieces stored between the MFMAs");
    W32Rows<D, NW> kr, vr;
    uint2 rp;                                             // ring_pos of row (thread % KB) of a ring block
    KeySeg br, nx;                                        // this block and the next
    auto fetch_pos = [&](const KeySeg& s) {
        // out-of-range offset (outside the ring) reads 0
        rp = buf_ld8(rpos, s.slot0 >= 0 ? (uint32_t)(s.slot0 + min((int)threadIdx.x % KB, min(s.count, KB) - 1)) * 8u
                                        : 0xFFFFFFF0u);
    };
    auto load_k = [&](const KeySeg& s, int j) { kr.load(s.kb, s.ks, min(s.count, KB) - 1, wv, lane, j); };
    auto load_v = [&](const KeySeg& s, int j) { vr.load(s.vb, s.vs, min(s.count, KB) - 1, wv, lane, j); };
    auto park_pos = [&](const KeySeg& s, int i) {
        if (threadIdx.x < KB) {
            const long kp = s.pos0 + threadIdx.x;
            bool val = (int)threadIdx.x < s.count;
            if (s.slot0 >= 0) val = val && (long)(((uint64_t)rp.y << 32) | rp.x) == kp;
            // sinks far behind the chunk clamp (always visible)
            sm.krel[i & 1][threadIdx.x] = val ? (int)max(kp - p_first, -(1L << 30)) : 0x7fffffff;
            const int nv = __popcll(__ballot(val));
            if (threadIdx.x == 0) sm.nval[i & 1] = nv;
        }
    };
    if (nblk > 0) {
        br = block_ref(0);
        fetch_pos(br);
#pragma unroll
        for (int j = 0; j < NCH; ++j) load_k(br, j);
#pragma unroll
        for (int j = 0; j < NCH; ++j) load_v(br, j);
#pragma unroll
        for (int j = 0; j < NCH; ++j) kr.park(sm.k, wv, lane, j);
        park_pos(br, 0);
    }
    const int trow = 4 * lg + (l16 >> 2), tcol = 4 * (l16 & 3);
    for (int i = 0; i < nblk; ++i) {
        lds_barrier();                                     // K_i is in LDS, V_{i-1} fully consumed
        // past the last block it is fetched and stored again: a condition would end in waits for the loads it joins
        nx = block_ref(min(i + 1, nblk - 1));
        fetch_pos(nx);
        // the pair's queries see something of the block: its first key is not past them all, its last one not behind
        // all of their windows
        const long k0 = br.pos0 - p_first, k1 = k0 + min(br.count, KB) - 1;
        const bool on = QW * pr < nq && k0 <= QW * pr + QW - 1 && (br.sink || QW * pr - k1 < a.W);
        const bool whole = !br.sink && k1 <= QW * pr && k0 > QW * pr + QW - 1 - (long)a.W &&
                           __builtin_amdgcn_readfirstlane(sm.nval[i & 1]) == KB;
        f32x4 s[QT][2];
        if (on) {
            // S^T = K Q^T for this block
#pragma unroll
            for (int qt = 0; qt < QT; ++qt) s[qt][0] = s[qt][1] = f32x4{0.f, 0.f, 0.f, 0.f};
            // step t: dims 32 (t / 2) .., key tile t % 2. The next step's fragment is read before this one's MFMAs; the
            // scheduling barriers keep the compiler from reading further ahead, into more registers than there are.
            auto read_k = [&](int t) {
                Planes f;
#pragma unroll
                for (int j = 0; j < 3; ++j) f.p[j] = ld16(&sm.k[j][16 * (t & 1) + l16][dh + 32 * (t >> 1) + 8 * lg]);
                return f;
            };
            Planes ak = read_k(0);
#pragma unroll
            for (int t = 0; t < 2 * NKD; ++t) {
                const Planes nk = read_k(min(t + 1, 2 * NKD - 1));
#pragma unroll
                for (int qt = 0; qt < QT; ++qt) mma3(s[qt][t & 1], ak, fq[qt][t >> 1]);
                if (t & 1)
#pragma unroll
                    for (int j = t / 2 * NP; j < (t / 2 + 1) * NP; ++j) {
                        vr.park(sm.v, wv, lane, j);
                        load_k(nx, j);
                    }
                ak = nk;
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int qt = 0; qt < QT; ++qt)
#pragma unroll
                for (int kt = 0; kt < 2; ++kt) sm.part[wv][2 * qt + kt][lane] = s[qt][kt];
        } else {
#pragma unroll
            for (int j = 0; j < NCH; ++j) {
                vr.park(sm.v, wv, lane, j);
                load_k(nx, j);
            }
        }
        lds_barrier();                                     // V_i is in LDS, K_i fully consumed
        if (on) {
#pragma unroll
            for (int qt = 0; qt < QT; ++qt)
#pragma unroll
                for (int kt = 0; kt < 2; ++kt) s[qt][kt] += sm.part[mate][2 * qt + kt][lane];
            Planes pb[QT];
            // Online softmax per query column, in the units of the products (the scale is in the exponent's FMA). A block
            // of whole keys inside every query's window needs no mask; else keys past wlow (qrel - W; sinks have no lower
            // end) up to the query's own position are kept.
            if (!whole) {
#pragma unroll
                for (int kt = 0; kt < 2; ++kt) {
                    const int4 kp = *reinterpret_cast<const int4*>(&sm.krel[i & 1][16 * kt + 4 * lg]);
                    const int kpe[4] = {kp.x, kp.y, kp.z, kp.w};
#pragma unroll
                    for (int qt = 0; qt < QT; ++qt) {
                        const int qp = qrel + 16 * qt, wlow = br.sink ? -0x7fffffff : max(qp - a.W, -0x7fffffff);
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            s[qt][kt][e] = (kpe[e] <= qp) & (kpe[e] > wlow) ? s[qt][kt][e] : -INFINITY;
                    }
                }
            }
#pragma unroll
            for (int qt = 0; qt < QT; ++qt) {
                float bm = s[qt][0][0];
#pragma unroll
                for (int e = 1; e < 8; ++e) bm = fmaxf(bm, s[qt][e / 4][e % 4]);
                const float mn = fmaxf(m[qt], lane_max4(bm)), mc = mn == -INFINITY ? 0.f : mn * scale2;
                const float corr = mn == -INFINITY ? 1.f : __builtin_amdgcn_exp2f((m[qt] - mn) * scale2);
                float ls = 0.f;
#pragma unroll
                for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[qt][kt][e], scale2, -mc));
                        s[qt][kt][e] = p;
                        ls += p;
                    }
                l[qt] = l[qt] * corr + lane_sum4(ls);
                m[qt] = mn;
                if (__any(corr != 1.f)) {
#pragma unroll
                    for (int dt = 0; dt < NDT; ++dt) {
                        o[qt][dt][0] *= corr; o[qt][dt][1] *= corr; o[qt][dt][2] *= corr; o[qt][dt][3] *= corr;
                    }
                }
                pb[qt] = split8<SPLIT_SMALL>(s[qt][0], s[qt][1]);      // (probabilities)
            }
            // O^T += V^T P^T: the K index 8 lg + e is key 4 lg + e of the first 16 (e < 4) or of the second
            auto read_v = [&](int dt) {
                Planes f;
#pragma unroll
                for (int j = 0; j < 3; ++j) {
                    const uint2 lo = lds_tr16(reinterpret_cast<const char*>(&sm.v[j][trow][dh + 16 * dt + tcol]));
                    const uint2 hi = lds_tr16(reinterpret_cast<const char*>(&sm.v[j][16 + trow][dh + 16 * dt + tcol]));
                    f.p[j] = make_uint4(lo.x, lo.y, hi.x, hi.y);
                }
                return f;
            };
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt) {
                const Planes av = read_v(dt);
#pragma unroll
                for (int qt = 0; qt < QT; ++qt) mma3(o[qt][dt], av, pb[qt]);
                if (dt & 1)
#pragma unroll
                    for (int j = dt / 2 * NP; j < (dt / 2 + 1) * NP; ++j) {
                        kr.park(sm.k, wv, lane, j);
                        load_v(nx, j);
                    }
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {
#pragma unroll
            for (int j = 0; j < NCH; ++j) {
                kr.park(sm.k, wv, lane, j);
                load_v(nx, j);
            }
        }
        park_pos(nx, i + 1);
        br = nx;
    }

    // epilogue: normalise, lse, gamma mix, store o [B][T][H][D]
    const float lnW = logf((float)a.W);
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
        const int qi = qrel + 16 * qt;
        if (qi >= nq) continue;
        const long tq = qi0 + qi;
        const float inv = 1.f / l[qt];
        const float lse = m[qt] * scale + logf(l[qt]);
        if (a.lse && lg == 0 && dh == 0) a.lse[((long)b * H + h) * a.T + tq] = lse;
        float gam = 0.f;
        if (a.mix_on && p_first + qi >= a.W)
            gam = 1.f / (1.f + __expf(-(a.z[((long)b * a.T + tq) * H + h] + a.mix_lse[h] * (lse - lnW))));
        const float ms = a.mix_on ? a.mem_scale[h] : 0.f;
        const long orow = (((long)b * a.T + tq) * H + h) * D + dh;
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
            for (int e = 0; e < 4; ++e) r4[e] = o[qt][dt][e] * inv;
            if (a.mix_on) {
                const float mv[4] = {om[dt].x, om[dt].y, om[dt].z, om[dt].w};
#pragma unroll
                for (int e = 0; e < 4; ++e) r4[e] = mixed ? r4[e] + gam * (ms * mv[e] - r4[e]) : r4[e];
            }
            if constexpr (BO) store4<BF16>(reinterpret_cast<uint16_t*>(a.o) + orow + d0, r4[0], r4[1], r4[2], r4[3]);
            else store4<F32>(reinterpret_cast<float*>(a.o) + orow + d0, r4[0], r4[1], r4[2], r4[3]);
        }
    }
}

template <int D, int NW>
static int launch_window(const WinArgs& args, hipStream_t stream) {
    WinArgs a = args;
    // the map counts 128-query items; 64-query ones are those of twice the length
    const int f = a.start < a.W ? 2 : 1;
    a.map = window_map_make(a.B, a.G, a.R, a.T * (8L / NW), f, 0);
    if (8 * a.map.per > 0x7fffffffL) return BF_STATUS_INVALID;
    const dim3 grid((unsigned)(8 * a.map.per)), block(64 * NW);
    if (a.o_dtype == DT_BF16) hipLaunchKernelGGL((window_kernel<D, NW, true>), grid, block, 0, stream, a);
    else hipLaunchKernelGGL((window_kernel<D, NW, false>), grid, block, 0, stream, a);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : (int)e;
}

// 64 or 128 queries per workgroup: 128 store each key block half as often; 64 make twice the workgroups, each with half the
// MFMAs of a block. 64 while every workgroup has a CU of its own (one wave per SIMD), where 128 would be half empty, and over
// short windows at the smaller dims, whose items are mostly their first loads and their ends. us a launch, 64 / 128 queries:
// 16 sequences of 20 queries, H = 16, D = 256, W = 2048 328 / 337; 200 of 20, D = 128, W = 64 149 / 282; 40 of 64, D = 128, W = 2048
// 489 / 674; 4096 queries, H = 16, W = 2048 D = 256 1299 / 746, D = 128 559 / 476; H = 32, D = 64 764 / 682; 16 of 300, W = 256,
// D = 256 319 / 256, D = 128 140 / 164, D = 64 (H = 32) 186 / 227; 3 of 2000, W = 512, D = 128 257 / 241, D = 64 (H = 8) 103 / 115.
// At D = 64 the 64-query form is for 32 queries or fewer over more than 128 keys (64 sequences of 20, H = 8, W = 256: 36 us against
// 43); otherwise the fp32 MFMAs on unsplit rows are faster (window_d64.hip).
template <int D>
static int launch_window_by_size(const WinArgs& a, hipStream_t stream) {
    const long keys = a.start + a.T < a.W ? a.start + a.T : a.W;
    const bool few = a.T <= 64 || (long)a.B * a.G * a.R * ((a.T + 63L) / 64) <= 256 || keys <= (D == 64 ? 1024 : D == 128 ? 256 : 0);
    if constexpr (D == 64)
        if (few && (a.T > 32 || keys <= 128) && a.B <= 65535 && (long)a.G * a.R <= 65535) return window_d64_dispatch(a, stream);
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
