// K2, fp32 operands, D = 64 and few queries or a short window: the sliding-window attention of window.hip on fp32 MFMAs.
//
// Reference: HybridAttention._window_fp32 (Heimdall/heimdall/hibrit.py:341-361) and the mix of :409-411; the visible keys, the
// softmax and the mix are those that window.hip states.
//
// At D = 64 a key block is little work beside the splitting of its rows into planes, unless 128 queries share it. One workgroup =
// 64 queries of one query head (4 waves x 16). Per block of 32 keys the K rows (row-major) and V rows (transposed) go to LDS as
// they are; the next block's are loaded into registers meanwhile. Scores are computed transposed (S^T = K Q^T), so each lane's
// softmax statistics belong to its own query column, and P feeds the P V product from registers. us a launch, planes / here: 4
// sequences of 1000 queries, H = 32, W = 64: 77 / 60; 16 of 300, W = 256 185 / 154; 3 of 2000, H = 8, W = 512 103 / 88; 40 of 64,
// H = 32, W = 2048 550 / 463.
#include "bf_common.h"
#include "bf_internal.h"

namespace bf {

namespace {

constexpr int D = 64, KB = 32, NT = 256, QW = 16, BQ = 4 * QW;      // head dim, keys per block, threads, queries per wave, per workgroup
constexpr int VEC = F32::VEC, KF = F32::KF, CPR = D / 4, KCH = KB * CPR / NT;

struct Shared {
    __align__(16) float ks[KB][D + VEC];     // key rows of the block
    float vt[D][KB + VEC];                   // value rows of the block, transposed [d][key]
    int krel[KB];                            // key position minus the workgroup's first query position; INT_MAX: not a key
};

// A run of key rows from one contiguous source (the sinks, the ring up to its wrap point, the ring after it, the chunk)
struct Seg {
    const float* kb;   // first key row
    const float* vb;   // first value row
    long ks, vs;       // row strides (elements)
    long pos0;         // position of the first row (sinks: 0)
    int count;         // rows
    int slot0;         // ring slot of the first row, or -1 outside the ring
    int sink;          // sink rows: visible to every query at or after their position, no window limit
};

struct Prefetch {
    f32x4 k[KCH];
    f32x4 v[4];        // a 4 x 4 block: keys 4 bt .., dims 4 bd ..
    uint2 rp;          // ring_pos of row (thread % KB) for ring blocks, read with the rows
};
constexpr int VBT = KB / 4, VBD = D / 4;
static_assert(VBT * VBD <= NT, "one value block per thread");

// Load the rows of one key block into registers. Rows past the segment's end are its last row again; their scores are masked
// (exec-masked loads would make the compiler wait for the whole prefetch early).
__device__ __forceinline__ void fetch(Prefetch& f, const Seg& br, rsrc_t rpos) {
    const int tid = threadIdx.x, last = min(br.count, KB) - 1;
    // out-of-range offset (outside the ring) reads 0
    f.rp = buf_ld8(rpos, br.slot0 >= 0 ? (uint32_t)(br.slot0 + min(tid % KB, last)) * 8u : 0xFFFFFFF0u);
#pragma unroll
    for (int j = 0; j < KCH; ++j) {
        const int c = tid + NT * j;
        f.k[j] = *reinterpret_cast<const f32x4*>(br.kb + min(c / CPR, last) * br.ks + 4 * (c % CPR));
    }
    const int bt = tid % VBT, bd = tid / VBT % VBD;
#pragma unroll
    for (int i = 0; i < 4; ++i) f.v[i] = *reinterpret_cast<const f32x4*>(br.vb + min(4 * bt + i, last) * br.vs + 4 * bd);
}

__device__ __forceinline__ void park(Shared& sm, const Prefetch& f, const Seg& br, long p_first) {
    const int tid = threadIdx.x;
#pragma unroll
    for (int j = 0; j < KCH; ++j) {
        const int c = tid + NT * j;
        *reinterpret_cast<f32x4*>(&sm.ks[c / CPR][4 * (c % CPR)]) = f.k[j];
    }
    if (tid < VBT * VBD) {
        const int bt = tid % VBT, bd = tid / VBT;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            *reinterpret_cast<f32x4*>(&sm.vt[4 * bd + i][4 * bt]) = f32x4{f.v[0][i], f.v[1][i], f.v[2][i], f.v[3][i]};
    }
    if (tid < KB) {
        const long kp = br.pos0 + tid;
        bool val = tid < br.count;
        if (br.slot0 >= 0) val = val && (long)(((uint64_t)f.rp.y << 32) | f.rp.x) == kp;
        sm.krel[tid] = val ? (int)max(kp - p_first, -(1L << 30)) : 0x7fffffff;   // sinks far behind the chunk clamp (always visible)
    }
}

template <bool BO>
__global__ __launch_bounds__(NT) void window_d64_kernel(WinArgs a) {
    constexpr int NKD = D / KF, NKT = KB / 16, NDT = D / 16, PF = KB / KF;
    __shared__ __align__(16) Shared sm;

    const int qb = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
    const int R = a.R, G = a.G, H = G * R, g = h / R;
    const int lane = lane_id(), wv = wave_id(), l16 = lane & 15, lg = lane >> 4;
    const long qi0 = (long)qb * BQ;                       // first query index of the workgroup
    const int nq = (int)min((long)BQ, (long)a.T - qi0);
    const long p_first = a.start + qi0, p_last = a.start + qi0 + nq - 1;
    const float scale = rsqrtf((float)D);

    const float* rk = a.ring_k ? reinterpret_cast<const float*>(a.ring_k) + ((long)b * G + g) * a.W * D : nullptr;
    const float* rv = a.ring_v ? reinterpret_cast<const float*>(a.ring_v) + ((long)b * G + g) * a.W * D : nullptr;
    const float* ck = reinterpret_cast<const float*>(a.k) + b * a.k_sb + g * a.k_sh;
    const float* cv = reinterpret_cast<const float*>(a.v) + b * a.v_sb + g * a.v_sh;

    // Q fragments (B operand of S^T = K Q^T): column l16, k range VEC lg of each KF step
    const int qp = QW * wv + l16;                         // query position minus p_first
    const float* qrow = reinterpret_cast<const float*>(a.q) + b * a.q_sb + h * a.q_sh + (qi0 + qp) * a.q_st;
    uint4 fq[NKD];
#pragma unroll
    for (int kf = 0; kf < NKD; ++kf) fq[kf] = qp < nq ? ld16(qrow + kf * KF + VEC * lg) : zero16();
    f32x4 o[NDT];
    float m = -INFINITY, l = 0.f;
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};

    // key segments, consumed in blocks of KB rows
    const long kp_lo = max((long)a.sinks, p_first - a.W + 1);
    Seg sg[4];
    int nb[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) sg[j] = Seg{ck, cv, 0, 0, 0, 0, -1, 0};
    if (a.n_sinks)
        sg[0] = Seg{reinterpret_cast<const float*>(a.sink_k) + ((long)b * G + g) * a.n_sinks * D,
                    reinterpret_cast<const float*>(a.sink_v) + ((long)b * G + g) * a.n_sinks * D, D, D, 0, a.n_sinks, -1, 1};
    const long rhi = min(p_last, a.start - 1);
    if (rk && kp_lo <= rhi) {
        const int sa = (int)(kp_lo % a.W);                // one division per workgroup
        const long n = rhi - kp_lo + 1, n1 = min(n, (long)(a.W - sa));
        sg[1] = Seg{rk + (long)sa * D, rv + (long)sa * D, D, D, kp_lo, (int)n1, sa, 0};
        if (n > n1) sg[2] = Seg{rk, rv, D, D, kp_lo + n1, (int)(n - n1), 0, 0};
    }
    const long clo = max(kp_lo, a.start);
    if (clo <= p_last)
        sg[3] = Seg{ck + (clo - a.start) * a.k_st, cv + (clo - a.start) * a.v_st, a.k_st, a.v_st, clo, (int)(p_last - clo + 1), -1, 0};
    int nblk = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        nb[j] = (sg[j].count + KB - 1) / KB;
        nblk += nb[j];
    }
    // block i as a segment of its own: the KB rows starting at row KB * (i - first block of its segment)
    auto block_ref = [&](int i) {
        Seg r = sg[3];
        int base = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (i >= base && i < base + nb[j]) {
                const int off = (i - base) * KB;
                r = sg[j];
                r.kb += off * sg[j].ks;
                r.vb += off * sg[j].vs;
                r.pos0 += off;
                r.count -= off;
                if (r.slot0 >= 0) r.slot0 += off;
            }
            base += nb[j];
        }
        return r;
    };

    const rsrc_t rpos = make_rsrc(a.ring_pos, a.ring_pos ? (uint32_t)a.W * 8u : 0u);
    Prefetch pf;
    Seg br;
    if (nblk > 0) {
        br = block_ref(0);
        fetch(pf, br, rpos);
    }
    for (int i = 0; i < nblk; ++i) {
        const bool sb = br.sink;
        __syncthreads();                                   // previous block fully consumed
        park(sm, pf, br, p_first);
        __syncthreads();
        if (i + 1 < nblk) {                                // uniform: the next block's loads fly during this one
            br = block_ref(i + 1);
            fetch(pf, br, rpos);
        }
        // S^T = K Q^T for this block
        f32x4 s[NKT];
#pragma unroll
        for (int kt = 0; kt < NKT; ++kt) s[kt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kf = 0; kf < NKD; ++kf)
#pragma unroll
            for (int kt = 0; kt < NKT; ++kt) mma<F32>(s[kt], ld16(&sm.ks[16 * kt + l16][kf * KF + VEC * lg]), fq[kf]);
        // mask, online softmax per query column
        const int wlow = sb ? -0x7fffffff : max(qp - a.W, -0x7fffffff);
        float bm = -INFINITY;
#pragma unroll
        for (int kt = 0; kt < NKT; ++kt) {
            const int4 kp = *reinterpret_cast<const int4*>(&sm.krel[16 * kt + 4 * lg]);
            const int kpe[4] = {kp.x, kp.y, kp.z, kp.w};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                s[kt][e] = (kpe[e] <= qp) & (kpe[e] > wlow) ? s[kt][e] * scale : -INFINITY;
                bm = fmaxf(bm, s[kt][e]);
            }
        }
        bm = fmaxf(bm, __shfl_xor(bm, 16));
        bm = fmaxf(bm, __shfl_xor(bm, 32));
        const float mn = fmaxf(m, bm), corr = mn == -INFINITY ? 1.f : __expf(m - mn);
        float ls = 0.f;
#pragma unroll
        for (int kt = 0; kt < NKT; ++kt)
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
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) {
            o[dt][0] *= corr; o[dt][1] *= corr; o[dt][2] *= corr; o[dt][3] *= corr;
        }
        // O^T += V^T P^T. P fragment f: keys KF f + 4 lg + e
#pragma unroll
        for (int f = 0; f < PF; ++f) {
            const uint4 pb = __builtin_bit_cast(uint4, s[f]);
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt) mma<F32>(o[dt], ld16(&sm.vt[16 * dt + l16][KF * f + 4 * lg]), pb);
        }
    }

    // epilogue: normalise, lse, gamma mix, store o [B][T][H][D]
    if (qp >= nq) return;
    const long tq = qi0 + qp;
    const float inv = 1.f / l, lse = m + logf(l);
    if (a.lse && lg == 0) a.lse[((long)b * H + h) * a.T + tq] = lse;
    float gam = 0.f;
    if (a.mix_on && p_first + qp >= a.W)
        gam = 1.f / (1.f + __expf(-(a.z[((long)b * a.T + tq) * H + h] + a.mix_lse[h] * (lse - logf((float)a.W)))));
    const float ms = a.mix_on ? a.mem_scale[h] : 0.f;
    const long orow = (((long)b * a.T + tq) * H + h) * D;
    // memory reads issued together (every row of o_mem exists); rows with gam = 0 keep the window output by selection, so rows
    // the delta rule never wrote cannot leak in
    const bool on = gam != 0.f;
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
            for (int e = 0; e < 4; ++e) r4[e] = on ? r4[e] + gam * (ms * mv[e] - r4[e]) : r4[e];
        }
        if constexpr (BO) store4<BF16>(reinterpret_cast<uint16_t*>(a.o) + orow + d0, r4[0], r4[1], r4[2], r4[3]);
        else store4<F32>(reinterpret_cast<float*>(a.o) + orow + d0, r4[0], r4[1], r4[2], r4[3]);
    }
}

}  // namespace

int window_d64_dispatch(const WinArgs& a, hipStream_t stream) {
    const dim3 grid((unsigned)((a.T + (long)BQ - 1) / BQ), (unsigned)(a.G * a.R), (unsigned)a.B);
    if (a.o_dtype == DT_BF16) hipLaunchKernelGGL((window_d64_kernel<true>), grid, dim3(NT), 0, stream, a);
    else hipLaunchKernelGGL((window_d64_kernel<false>), grid, dim3(NT), 0, stream, a);
    return (int)hipGetLastError();
}

}  // namespace bf
