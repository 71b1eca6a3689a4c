// The split attend: attend_two_pass (ops/attention.py:429-449) of one query per sequence in two
// launches that wait on nobody, bit-exact with the reference.
//
// score_max_kernel scores every token and keeps only the maximum of each 64-token block and of each
// workgroup's blocks, per query head. In the decode step it also rotates the wire rows and encodes
// and appends the new one. The maximum of a sequence is then known to every workgroup of the second
// launch from a few hundred words.
//
// sum_kernel gives a workgroup up to 64 consecutive blocks. A block none of whose tokens comes within
// delta_max of the maximum contributes nothing (every p is 0) and is skipped: of a peaked softmax
// nearly all are. The others, in turn a wave, are scored again (a score is cheaper to compute twice
// than eight bytes a token and head are to store and load) and summed on the matrix cores. The last
// workgroup of a (sequence, KV head) adds up the workgroups' sums, in 64 bits, clamps and divides; a
// head whose scores are not exact is recomputed on the serial path (serial_head.h).
//
// Matrix operands. Scores: a query head's four balanced digits are four rows, so 4 heads fill the 16
// rows (8 heads: two sets), against 16 tokens' centroid digits, three products a 64 channels; the
// result has lane = (token, head) with the row digits in its four registers. There p and w = v_norm p
// are computed, one token a lane and head. Sums: lane = (head, digit) takes w of four tokens, and one
// fma a value code leaves that digit of floor(w c_v / 2^23) in a byte of the fp64 mantissa; times the
// one-hot value codes of 16 channels this gives lane = (head, digit) four channels' sums of that
// digit, exact in int32 over a workgroup's 4,096 tokens.
//
// Bounds: up to some 4,096 tokens a chain, latency (a wave alone on its SIMD, instructions that no
// wave before it fetched): 11 us a launch, whatever the length. A two-pass decode step of 4,097
// tokens at d = 64, 8 KV heads: 23.2 us (75.0 as a write, a maximum and a summing launch of 1,024
// tokens a workgroup in fp64). Beyond, the matrix products and the digits' extraction: a flat softmax
// over 16 x 32,768 tokens 213 us (833), of 131,072 tokens 98 us (281).
#include <algorithm>
#include <cstdlib>

#include "digits.h"
#include "query.h"
#include "row_codec.h"
#include "serial_head.h"
#include "wave.h"

namespace insitu {
namespace sp {

constexpr int BT = 64;                  // tokens a block
constexpr int W = 4;                    // waves a workgroup
constexpr int MAXU = 16;                // blocks a wave of sum_kernel, at most
constexpr int MAXWG = 64;               // workgroups of sum_kernel a chain, at most: a lane each
constexpr uint32_t LUT_N = LUT_SPAN + 1;
constexpr double TERM_MAGIC = 402653184.0 + 8421504.0;   // 1.5 * 2^28 + 0x808080: ulp 2^-24
constexpr int32_t TOP_BYTE = -72;       // digit 3's byte for 0: 0xB8, exponent bits of the magic number above it
constexpr double BIG_Q = 0x1p46;        // ||q||_1 max|c| from which dot / 2^16 may not fit int32
constexpr uint64_t RUN = 1ull << 63;    // meta: the workgroup has sums

__device__ __forceinline__ void pub64(void *p, uint64_t v) {
    __hip_atomic_store((uint64_t *)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint64_t get64(const void *p) {
    return __hip_atomic_load((uint64_t *)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void stores_done() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_waitcnt(0x0F70);          // vmcnt(0)
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// Maximum and sum over a row of 16 lanes, in every lane of it.
__device__ __forceinline__ int64_t row_max64(int64_t v) {
    v = OpMax64::f(v, dpp64<DPP_QUAD_1032>(v, v));
    v = OpMax64::f(v, dpp64<DPP_QUAD_2301>(v, v));
    v = OpMax64::f(v, dpp64<DPP_ROW_HALF_MIRROR>(v, v));
    return OpMax64::f(v, dpp64<DPP_ROW_MIRROR>(v, v));
}
__device__ __forceinline__ uint32_t row_sum32(uint32_t v) {
    v += dpp32<DPP_QUAD_1032>(0u, v);
    v += dpp32<DPP_QUAD_2301>(0u, v);
    v += dpp32<DPP_ROW_HALF_MIRROR>(0u, v);
    return v + dpp32<DPP_ROW_MIRROR>(0u, v);
}

// The scratch of a cache: for GP padded heads (4 or 8) a chain.
struct Scratch {
    uint32_t *done;       // [chain]: workgroups done with their runs (zero between attends)
    uint32_t *qbad;       // [chain]: heads whose scores may not be exact, a bit each
    int32_t *qr;          // [chain][GP][d]: the rotated query rows
    int64_t *bm;          // [chain][GP][nblk]: block maxima
    int64_t *cm;          // [chain][GP][nblk / 4]: the maxima of score_max_kernel's workgroups
    uint64_t *meta;       // [chain][GP][workgroup of sum_kernel]: sum of p, RUN
    int64_t *S;           // [chain][GP][workgroup][d]: sums of floor(v_norm p c / 2^23)
    int32_t nblk, nwg;
};

// A lane's key codes of one tile: channels [grp d / 4, (grp + 1) d / 4) of token t.
template <int D, int KB>
struct Codes {
    static constexpr int N = KB == 4 ? D / 32 : KB == 3 ? (D == 64 ? 2 : 3) : D / 64;
    uint32_t w[N];
    __device__ __forceinline__ void load(const uint8_t *hb, int64_t span, int64_t t, int grp) {
        if constexpr (KB == 4 && D == 64) {
            const uint2 v = *(const uint2 *)(hb + (grp >> 1) * span + t * 16 + (grp & 1) * 8);
            w[0] = v.x;
            w[1] = v.y;
        } else if constexpr (KB == 4) {
            const uint4 v = *(const uint4 *)(hb + grp * span + t * 16);
            w[0] = v.x;
            w[1] = v.y;
            w[2] = v.z;
            w[3] = v.w;
        } else if constexpr (KB == 3) {
            const int d0 = D == 64 ? (3 * grp) >> 1 : 3 * grp;
#pragma unroll
            for (int i = 0; i < N; ++i) {
                const int dw = d0 + i, p = dw >> 2;              // d = 64: 6 words, the second plane 8 bytes wide
                w[i] = *(const uint32_t *)(hb + p * span + t * (D == 64 && p == 1 ? 8 : 16) + (dw & 3) * 4);
            }
        } else if constexpr (D == 64) {
            w[0] = *(const uint32_t *)(hb + t * 16 + grp * 4);
        } else {
            const uint2 v = *(const uint2 *)(hb + (grp >> 1) * span + t * 16 + (grp & 1) * 8);
            w[0] = v.x;
            w[1] = v.y;
        }
    }
    // the 16 codes of block b
    __device__ __forceinline__ uint64_t bits(int b, int grp) const {
        if constexpr (KB == 4)
            return (uint64_t)w[2 * b] | (uint64_t)w[2 * b + 1] << 32;
        else if constexpr (KB == 3 && D == 64)
            return ((uint64_t)w[0] | (uint64_t)w[1] << 32) >> (16 * (grp & 1));
        else if constexpr (KB == 3)
            return b == 0 ? (uint64_t)w[0] | (uint64_t)w[1] << 32 : ((uint64_t)w[1] | (uint64_t)w[2] << 32) >> 16;
        else
            return w[b];
    }
};

// The query operand from rotated rows in LDS: row = (head 4 s + l / 4, digit l % 4).
template <int D, int KB>
__device__ __forceinline__ void query_operand(const int32_t (*qi)[D], int s, int lane, v4i (&a)[D / 64]) {
    const int32_t *row = qi[4 * s + ((lane & 15) >> 2)];
    const int sh = 8 * (lane & 3), c0 = (lane >> 4) * (D / 4);
#pragma unroll
    for (int b = 0; b < D / 64; ++b)
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            uint32_t o = 0;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                o |= ((balanced(row[c0 + 16 * b + channel_of(KB, 4 * w + j)]) >> sh) & 0xFFu) << (8 * j);
            a[b][w] = (int)o;
        }
}

// floor(dot k_norm / 2^24) of a tile's token (lane % 16) and head (lane / 16) of set s: dot the sum
// over the row digits (registers) and centroid digits (l) of T[l], as int64 arithmetic wraps.
__device__ __forceinline__ int64_t score_of(const v4i (&T)[3], int32_t kn, bool big) {
    const int32_t a0 = T[0][0], a1 = T[0][1] + T[1][0], a2 = T[0][2] + T[1][1] + T[2][0];
    const int32_t a3 = T[0][3] + T[1][2] + T[2][1], a4 = T[1][3] + T[2][2], a5 = T[2][3];
    if (big) {
        int64_t dot = a5;
        dot = wadd(wmul(dot, 256), a4);
        dot = wadd(wmul(dot, 256), a3);
        dot = wadd(wmul(dot, 256), a2);
        dot = wadd(wmul(dot, 256), a1);
        dot = wadd(wmul(dot, 256), a0);
        return wmul(dot, kn) >> (CENT_FRAC + 9);
    }
    const int32_t lo = a0 + (a1 << 8);
    const int32_t hi = (int32_t)((uint32_t)a2 + ((uint32_t)a3 << 8) + ((uint32_t)a4 << 16) + ((uint32_t)a5 << 24));
    return ((int64_t)hi * kn + (((int64_t)lo * kn) >> 16)) >> 8;
}

template <int D, int KB, int NS>
struct ScoreLds {
    int32_t qi[4 * NS][D];
    alignas(16) uint32_t dig[3][4];
    int64_t wm[W][4 * NS];              // each wave's maxima
    int64_t lastm[4 * NS];              // the last block's, without the new token
    int64_t kc[16];
    int64_t bnd[2][255];                // the new row: boundaries, codes, norms
    uint8_t codes[2][MAX_D];
    int64_t nn[2];
    uint32_t bad;                       // heads whose scores may not be exact
    int big;
    unsigned long long mabs;
};

// Grid: chains fastest. Workgroup x of a chain takes 4 r blocks from 4 r x on. STEP: the decode step
// (si; len holds the lengths before it); else the caller's rotated rows q.
template <int D, int KB, int NS, bool STEP>
__global__ void __launch_bounds__(W * 64) score_max_kernel(Geom g, const Tables *__restrict__ tabs,
                                                          const int32_t *__restrict__ q, const int64_t *__restrict__ len,
                                                          Scratch sc, int r, DevStats *st, StepIn si) {
    __shared__ ScoreLds<D, KB, NS> S;
    constexpr int CPL = D / 64, GP = 4 * NS;
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 15, grp = lane >> 4, G = g.G;
    const int n_chains = g.batch * g.n_kv;
    const int chain = (int)(blockIdx.x % (unsigned)n_chains), x = (int)(blockIdx.x / (unsigned)n_chains);
    const int b = chain / g.n_kv, kvh = chain % g.n_kv;
    const int64_t T0 = len[b], T = T0 + (STEP ? 1 : 0);          // T0: the rows in memory
    const int nblk = (int)((T + BT - 1) / BT);
    if (x > 0 && 4 * r * x >= nblk) return;
    const bool owner = STEP && x == (nblk - 1) / (4 * r);        // this workgroup holds the new token
    if (STEP && x == 0 && kvh == 0 && tid == 0) si.len_out[b] = T;

    // -- the small loads, then the first block's rows -----------------------------------------
    const int64_t kc_t = tid < (1 << g.kb) ? tabs->kc[tid] : 0;
    int32_t qv[NS][CPL], kvv[CPL];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const int h = 4 * s + wv;
#pragma unroll
        for (int k = 0; k < CPL; ++k) qv[s][k] = 0;
        if (h < G) load_vec<CPL>((STEP ? si.qw : q) + ((int64_t)b * g.n_q + kvh * G + h) * D, D, qv[s]);
    }
    if (owner && wv < 2) load_vec<CPL>((wv == 0 ? si.kw : si.vw) + ((int64_t)b * g.n_kv + kvh) * D, D, kvv);
    if (owner) stage_bounds(tabs, g, S.bnd);
    const double cmax = tabs->kc_absmax;
    const uint8_t *hb = plane_ptr(g, b, kvh, 0), *nb = hb + (g.n_planes - 1) * g.span;
    Codes<D, KB> cur[4], nxt[4];
    uint32_t cn[4], nn[4];
    auto load = [&](int blk, Codes<D, KB> (&c)[4], uint32_t (&n)[4]) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            int64_t t = (int64_t)blk * BT + 16 * j + col;
            t = t < T0 ? t : T0 > 0 ? T0 - 1 : 0;      // (row 0 lies in the cache whatever its length)
            c[j].load(hb, g.span, t, grp);
            n[j] = *(const uint32_t *)(nb + t * 4);
        }
    };
    const int blk0 = 4 * r * x + wv;
    if (blk0 < nblk) load(blk0, nxt, nn);
    if (tid == 0) {
        S.bad = 0;
        S.big = 0;
        S.mabs = 0;
    }
    if (tid < 16) {
        S.kc[tid] = kc_t;
        const uint32_t z = balanced((int32_t)kc_t);
#pragma unroll
        for (int l = 0; l < 3; ++l) ((uint8_t *)S.dig[l])[tid] = (uint8_t)(z >> (8 * l));
    }
    __syncthreads();
    // -- the query rows: rotated, bounded, staged -----------------------------------------
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const int h = 4 * s + wv;
        if (STEP && h < G) rotate_loaded<CPL>(qv[s], D, si.rounds, si.sg, qv[s], x == 0 ? &st->range_errors : nullptr);
        int64_t l1 = 0;
        uint32_t big = 0, out = 0;
#pragma unroll
        for (int k = 0; k < CPL; ++k) {
            const uint32_t a = qv[s][k] < 0 ? 0u - (uint32_t)qv[s][k] : (uint32_t)qv[s][k];
            S.qi[h][lane + 64 * k] = qv[s][k];
            if (x == 0) sc.qr[((int64_t)chain * GP + h) * D + lane + 64 * k] = qv[s][k];
            l1 += a;
            out += a >= (uint32_t)Q_ROT_LIMIT ? 1 : 0;
            big |= a >> 30;
        }
        const double bq = (double)wave_sum_i64(l1) * cmax;
        if (lane == 0 && (!(bq < DOT_LIMIT))) atomicOr(&S.bad, 1u << h);
        if (big) atomicOr(&S.bad, 1u << h);
        if (lane == 0 && !(bq < BIG_Q)) S.big = 1;
        if (x == 0 && out) atomicAdd(&st->range_errors, (unsigned long long)out);
    }
    __syncthreads();
    if (x == 0 && tid == 0) sc.qbad[chain] = S.bad | (S.big ? 0x80000000u : 0u);
    const bool big = uni32(S.big);
    const uint32_t badm = (uint32_t)uni32((int)S.bad);
    if (owner && wv < 2) {
        // the new row's key (wave 0) and value; it is scored from its codes below
        rotate_loaded<CPL>(kvv, D, si.rounds, si.sg, kvv, &st->range_errors);
        int64_t v[CPL];
#pragma unroll
        for (int k = 0; k < CPL; ++k) v[k] = kvv[k];
        const int64_t n = encode_field<CPL>(v, D, g.norm_frac, S.bnd[wv], (1 << (wv == 0 ? g.kb : g.vb)) - 1, S.codes[wv]);
        if (lane == 0) S.nn[wv] = n;
    }

    // -- scores ---------------------------------------------------------------------------
    v4i qa[NS][CPL];
#pragma unroll
    for (int s = 0; s < NS; ++s) query_operand<D, KB>(S.qi, s, lane, qa[s]);
    uint32_t dg[3][4];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) dg[i][j] = S.dig[i][j];
    int64_t mabs = 0, wm[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) wm[s] = SCORE_LO;
    for (int i = 0; i < r; ++i) {
        const int blk = blk0 + 4 * i;
        if (blk >= nblk) break;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            cur[j] = nxt[j];
            cn[j] = nn[j];
        }
        if (i + 1 < r && blk + 4 < nblk) load(blk + 4, nxt, nn);
        int64_t mx[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) mx[s] = SCORE_LO;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            v4i T3[NS][3];
#pragma unroll
            for (int s = 0; s < NS; ++s)
#pragma unroll
                for (int l = 0; l < 3; ++l) T3[s][l] = v4i{0, 0, 0, 0};
#pragma unroll
            for (int k = 0; k < CPL; ++k) {
                v4i o[3];
                expand16<KB>(cur[j].bits(k, grp), dg, o);
#pragma unroll
                for (int s = 0; s < NS; ++s)
#pragma unroll
                    for (int l = 0; l < 3; ++l) T3[s][l] = mma(qa[s][k], o[l], T3[s][l]);
            }
            const int32_t kn = (int16_t)(uint16_t)cn[j];
            const bool in = (int64_t)blk * BT + 16 * j + col < T0;
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                const int64_t v = score_of(T3[s], kn, big);
                const int64_t a = v < 0 ? -v : v;
                mabs = in && a > mabs && 4 * s + grp < G && !(badm >> (4 * s + grp) & 1) ? a : mabs;
                mx[s] = in && v > mx[s] ? v : mx[s];
            }
        }
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            mx[s] = row_max64(mx[s]);
            wm[s] = mx[s] > wm[s] ? mx[s] : wm[s];
            if (col == 0) {
                if (owner && blk == nblk - 1)
                    S.lastm[4 * s + grp] = mx[s];
                else
                    sc.bm[((int64_t)chain * GP + 4 * s + grp) * sc.nblk + blk] = mx[s];
            }
        }
    }
#pragma unroll
    for (int s = 0; s < NS; ++s)
        if (col == 0) S.wm[wv][4 * s + grp] = wm[s];
    mabs = wave_max_i64(mabs);
    if (lane == 0) atomicMax(&S.mabs, (unsigned long long)mabs);
    __syncthreads();
    // the workgroup's maxima, with the new token's scores: a wave a head, lane = channel
    for (int h = wv; h < GP; h += W) {
        int64_t m = S.wm[0][h];
#pragma unroll
        for (int w = 1; w < W; ++w) m = S.wm[w][h] > m ? S.wm[w][h] : m;
        if (owner) {
            int64_t dot = 0;
#pragma unroll
            for (int k = 0; k < CPL; ++k) dot = wadd(dot, wmul(S.qi[h][lane + 64 * k], S.kc[S.codes[0][lane + 64 * k]]));
            const int64_t v = wmul(wave_sum_i64(dot), S.nn[0]) >> (CENT_FRAC + 9);
            const int64_t a = v < 0 ? -v : v;
            if (lane == 0 && h < G && !(badm >> h & 1)) atomicMax(&S.mabs, (unsigned long long)a);
            const int64_t lm = v > S.lastm[h] ? v : S.lastm[h];
            if (lane == 0) sc.bm[((int64_t)chain * GP + h) * sc.nblk + nblk - 1] = lm;
            m = v > m ? v : m;
        }
        if (lane == 0) sc.cm[((int64_t)chain * GP + h) * ((sc.nblk + 3) / 4) + x] = m;
    }
    if (owner && wv == W - 1 && lane < g.row_bytes / 4)
        *row_word_ptr(g, b, kvh, T - 1, lane) = pack_row_word(g, S.codes, S.nn[0], S.nn[1], lane);
    __syncthreads();
    if (tid == 0 && S.mabs > st->max_abs_score) atomicMax(&st->max_abs_score, S.mabs);
}

template <int D, int KB, int NC, int NS>
struct SumLds {
    static constexpr int GP = 4 * NS, VW = (D * (NC == 8 ? 3 : 2)) / 32;
    static constexpr int RS = D == 64 ? 60 : 116;
    union {
        struct {
            int32_t qi[GP][D];
            uint32_t vraw[W][16][VW];           // a tile's value words, a wave
            int32_t c9[8];                      // value centroids << 9
            int32_t Sm[2][GP][D];               // the workgroup's sums: digits 0 and 1, 2 and 3
            uint16_t lut[LUT_N + 7];
        } m;
        SerialLds<RS> fb[W];
    } u;
    alignas(16) uint32_t dig[3][4];
    int64_t mx[GP];
    unsigned long long act[GP];                 // the workgroup's blocks that contribute, a bit each
    uint32_t Lm[GP];
    unsigned long long macc, aovf;
    uint32_t bad;
    int last;
};

// Grid: chains fastest. Workgroup x of a chain takes 4 ub blocks from 4 ub x on.
template <int D, int KB, int NC, int NS>
__global__ void __launch_bounds__(W * 64, 2) sum_kernel(Geom g, const Tables *__restrict__ tabs, int32_t *out,
                                                       const int64_t *__restrict__ len, Scratch sc, int r, int ub,
                                                       DevStats *st) {
    using L = SumLds<D, KB, NC, NS>;
    __shared__ L S;
    constexpr int CPL = D / 64, GP = 4 * NS, CT = D / 16, PVK = NC / 4, VW = L::VW, VQ = (VW + 3) / 4;
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 15, grp = lane >> 4, G = g.G;
    const int hh = col >> 2, dgt = col & 3;            // the sums' lane: head 4 s + hh, digit
    const int n_chains = g.batch * g.n_kv;
    const int chain = (int)(blockIdx.x % (unsigned)n_chains), x = (int)(blockIdx.x / (unsigned)n_chains);
    const int b = chain / g.n_kv, kvh = chain % g.n_kv;
    const int64_t T = len[b];
    const int nblk = (int)((T + BT - 1) / BT), fb = 4 * ub * x;      // the workgroup's first block
    if (x > 0 && fb >= nblk) return;
    const int nwg = nblk > 0 ? (nblk + 4 * ub - 1) / (4 * ub) : 1;
    const int64_t crow = (int64_t)chain * GP;
    const uint32_t qb = sc.qbad[chain];
    const bool big = uni32((int)(qb >> 31));
    const int64_t delta_max = tabs->delta_max;

    // -- the maximum of all, and the blocks that contribute -----------------------------------
    const int nc1 = (sc.nblk + 3) / 4;
    for (int h = wv; h < GP; h += W) {
        const int64_t *bm = sc.bm + (crow + h) * sc.nblk, *cm = sc.cm + (crow + h) * nc1;
        const int blk = fb + lane;
        const bool in = lane < 4 * ub && blk < nblk;
        const int64_t own = in ? bm[blk] : SCORE_LO;
        const int end = (nblk + 4 * r - 1) / (4 * r);
        int64_t m = SCORE_LO;
        for (int i = lane; i < end; i += 256) {
            int64_t v[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) v[k] = i + 64 * k < end ? cm[i + 64 * k] : SCORE_LO;
#pragma unroll
            for (int k = 0; k < 4; ++k) m = v[k] > m ? v[k] : m;
        }
        m = wave_max_i64(m);
        const unsigned long long act = __ballot(in && h < G && own > m - delta_max);
        if (lane == 0) {
            S.mx[h] = m;
            S.act[h] = act;
        }
    }
    if (tid == 0) {
        S.macc = S.aovf = 0;
        S.bad = 0;
    }
    if (tid < GP) S.Lm[tid] = 0;
    __syncthreads();
    unsigned long long any = 0;
#pragma unroll
    for (int h = 0; h < GP; ++h) any |= S.act[h];
    if (any) {
        const int32_t ex = tabs->exp_table[tid];
        const int32_t kc = tid < (1 << g.kb) ? (int32_t)tabs->kc[tid] : 0;
        const int32_t vc = tid < (1 << g.vb) ? (int32_t)tabs->vc[tid] : 0;
        for (int i = tid; i < GP * D; i += W * 64) ((int32_t *)S.u.m.qi)[i] = sc.qr[crow * D + i];
#pragma unroll
        for (int i = 0; i < LUT_SPAN / 256; ++i) S.u.m.lut[256 * i + tid] = (uint16_t)(ex >> i);
        if (tid == 0) S.u.m.lut[LUT_SPAN] = 0;
        if (tid < 8) S.u.m.c9[tid] = vc << 9;
        if (tid < 16) {
            const uint32_t z = balanced(kc);
#pragma unroll
            for (int l = 0; l < 3; ++l) ((uint8_t *)S.dig[l])[tid] = (uint8_t)(z >> (8 * l));
        }
        for (int i = tid; i < 2 * GP * D; i += W * 64) ((int32_t *)S.u.m.Sm)[i] = 0;
        __syncthreads();
    }

    // -- this wave's blocks: every W-th of those that contribute ------------------------------
    unsigned long long left = any;
    for (int k = 0; k < wv; ++k) left &= left - 1;
    if (left) {
        double vcs[NC];
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            vcs[i] = (double)uni32(S.u.m.c9[i]) * 0x1p-32;           // value centroids / 2^23
            vcs[i] = __longlong_as_double(uni64(__double_as_longlong(vcs[i])));
        }
        v4i Sd[NS][CT];                                // a digit's sums
        uint32_t lp[NS];                               // lane = (token, head): sum of p
        int64_t m[NS];
        int32_t noff = 0;                              // products in Sd: digit 3's offset
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            lp[s] = 0;
            m[s] = S.mx[4 * s + grp];
#pragma unroll
            for (int c = 0; c < CT; ++c) Sd[s][c] = v4i{0, 0, 0, 0};
        }
        v4i qa[NS][CPL];
#pragma unroll
        for (int s = 0; s < NS; ++s) query_operand<D, KB>(S.u.m.qi, s, lane, qa[s]);
        uint32_t dg[3][4];
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) dg[i][j] = S.dig[i][j];
        const uint8_t *hb = plane_ptr(g, b, kvh, 0), *nb = hb + (g.n_planes - 1) * g.span;
        const int kpl = (g.key_bytes + 15) / 16, vwords = g.value_bytes / 4;
        // the byte of a term that is this lane's digit, for each of 4 codes in turn
        const uint32_t bsel = dgt == 0 ? 3u : 3u + (uint32_t)dgt;            // low word byte 3; high word bytes 0, 1, 2
        const uint32_t flip = dgt == 3 ? 0u : 0x80808080u;
        Codes<D, KB> cd;
        uint32_t nw, vr[VQ];
        // a tile's rows: lane = (token, quarter of the key field and of the value words)
        auto load = [&](int64_t t) __attribute__((always_inline)) {
            t += col;
            t = t < T ? t : T - 1;
            cd.load(hb, g.span, t, grp);
            nw = *(const uint32_t *)(nb + t * 4);
#pragma unroll
            for (int i = 0; i < VQ; ++i) {
                const int w = grp + 4 * i, p = w >> 2;
                const int width = g.value_bytes - 16 * p < 16 ? g.value_bytes - 16 * p : 16;
                vr[i] = w < vwords ? *(const uint32_t *)(hb + (kpl + p) * g.span + t * width + (w & 3) * 4) : 0u;
            }
        };
        // tile j of block lb, and behind it the next one
        auto next = [&]() __attribute__((always_inline)) {
            const int i = __ffsll((long long)left) - 1;
#pragma unroll
            for (int k = 0; k < W; ++k) left &= left - 1;
            return i;
        };
        int lb = next(), j = 0;
        load((int64_t)(fb + lb) * BT);
        for (bool done = false; !done;) {
            const int64_t t0 = (int64_t)(fb + lb) * BT + 16 * j;
            const Codes<D, KB> cc = cd;
            const uint32_t cw = nw;
            uint32_t cv[VQ];
#pragma unroll
            for (int i = 0; i < VQ; ++i) cv[i] = vr[i];
            if (j < 3 && t0 + 16 < T) {
                ++j;
            } else if (left) {
                lb = next();
                j = 0;
            } else {
                done = true;
            }
            if (!done) load((int64_t)(fb + lb) * BT + 16 * j);
            v4i T3[NS][3];
#pragma unroll
            for (int s = 0; s < NS; ++s)
#pragma unroll
                for (int l = 0; l < 3; ++l) T3[s][l] = v4i{0, 0, 0, 0};
#pragma unroll
            for (int k = 0; k < CPL; ++k) {
                v4i o[3];
                expand16<KB>(cc.bits(k, grp), dg, o);
#pragma unroll
                for (int s = 0; s < NS; ++s)
#pragma unroll
                    for (int l = 0; l < 3; ++l) T3[s][l] = mma(qa[s][k], o[l], T3[s][l]);
            }
            const int32_t kn = (int16_t)(uint16_t)cw, vn = (int16_t)(uint16_t)(cw >> 16);
            uint32_t p[NS], some = 0;
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                const uint64_t dl = (uint64_t)(m[s] - score_of(T3[s], kn, big));
                const uint32_t i = dl < (uint64_t)delta_max ? (uint32_t)dl : (uint32_t)delta_max;
                p[s] = t0 + col < T && 4 * s + grp < G ? S.u.m.lut[__umulhi(i, (uint32_t)LOG2E_Q16 << 8)] : 0u;
                some |= p[s];
            }
            if (__ballot(some != 0) == 0) continue;
            // the tile's value codes: lane = (channel, 4 tokens), one-hot
            wave_sync();
#pragma unroll
            for (int i = 0; i < VQ; ++i)
                if (VW % 4 == 0 || grp + 4 * i < VW) S.u.m.vraw[wv][col][grp + 4 * i] = cv[i];
            wave_sync();
            v4i oh[CT][PVK];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const uint32_t *row = S.u.m.vraw[wv][4 * grp + k];
#pragma unroll
                for (int c = 0; c < CT; ++c) {
                    if constexpr (NC == 4) {
                        const int bit = (16 * c + col) * g.vb;
                        oh[c][0][k] = (int)(1u << (8 * ((row[bit >> 5] >> (bit & 31)) & ((1u << g.vb) - 1u))));
                    } else {
                        const int bit = (16 * c + col) * 3, w = bit >> 5;
                        const uint32_t hi = row[w + 1 < VW ? w + 1 : w];
                        const uint64_t h = 1ull << (8 * (__builtin_amdgcn_alignbit(hi, row[w], bit & 31) & 7u));
                        oh[c][k >> 1][2 * (k & 1)] = (int)(uint32_t)h;
                        oh[c][k >> 1][2 * (k & 1) + 1] = (int)(uint32_t)(h >> 32);
                    }
                }
            }
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                lp[s] += p[s];
                const int32_t w = __mul24(vn, (int)p[s]);
                v4i B[PVK];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const double wd = (double)__shfl(w, hh * 16 + 4 * grp + k);
#pragma unroll
                    for (int q4 = 0; q4 < NC / 4; ++q4) {
                        uint32_t o = 0;
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const uint64_t y = (uint64_t)__double_as_longlong(fma(wd, vcs[4 * q4 + e], TERM_MAGIC));
                            const uint32_t sel = (0x0C0C0C0Cu & ~(0xFFu << (8 * e))) | bsel << (8 * e);
                            o |= perm((uint32_t)(y >> 32), (uint32_t)y, sel);
                        }
                        B[NC == 4 ? 0 : k >> 1][NC == 4 ? k : 2 * (k & 1) + q4] = (int)(o ^ flip);
                    }
                }
#pragma unroll
                for (int c = 0; c < CT; ++c)
#pragma unroll
                    for (int k = 0; k < PVK; ++k) Sd[s][c] = mma(oh[c][k], B[k], Sd[s][c]);
            }
            ++noff;
        }
        // -- into the workgroup's sums: digits 0 and 1 together, and 2 and 3 ----------------------
        const int off = dgt == 3 ? TOP_BYTE * 16 * noff : 0, sh = 8 * (dgt & 1);
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const uint32_t l = row_sum32(lp[s]);
            if (col == 0) atomicAdd(&S.Lm[4 * s + grp], l);
            int32_t *to = &S.u.m.Sm[dgt >> 1][4 * s + hh][4 * grp];
#pragma unroll
            for (int c = 0; c < CT; ++c)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int32_t v = (int32_t)((uint32_t)(Sd[s][c][i] - off) << sh);
                    const int32_t both = v + (int32_t)dpp32<DPP_QUAD_1032>(0u, (uint32_t)v);
                    if ((dgt & 1) == (i & 1)) atomicAdd(to + 16 * c + i, both);
                }
        }
    }
    __syncthreads();
    // -- publish, a wave a head; then the chain's last workgroup adds up ------------------------------
    for (int h = wv; h < G; h += W) {
        const int64_t at = (crow + h) * sc.nwg + x;
        if (any) {
#pragma unroll
            for (int k = 0; k < CPL; ++k) {
                const int c = lane + 64 * k;
                pub64(sc.S + at * D + c, (uint64_t)(S.u.m.Sm[0][h][c] + (int64_t)S.u.m.Sm[1][h][c] * 65536));
            }
        }
        if (lane == 0) pub64(sc.meta + at, any ? RUN | S.Lm[h] : 0ull);
    }
    stores_done();
    __syncthreads();
    if (tid == 0) {
        const uint32_t n = __hip_atomic_fetch_add(sc.done + chain, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        S.last = n == (uint32_t)(nwg - 1);
        if (S.last) __hip_atomic_store(sc.done + chain, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!S.last) return;

    for (int h = wv; h < G; h += W) {
        if (qb >> h & 1) {
            if (lane == 0) atomicOr(&S.bad, 1u << h);
            continue;
        }
        const int64_t base = (crow + h) * sc.nwg;
        const uint64_t mt = lane < nwg ? get64(sc.meta + base + lane) : 0ull;
        unsigned long long runs = __ballot((mt & RUN) != 0);
        const int64_t l = wave_sum_i64((int64_t)(mt & ~RUN));
        int64_t acc[CPL];
#pragma unroll
        for (int k = 0; k < CPL; ++k) acc[k] = 0;
        constexpr int RB = 16 / CPL;
        while (runs) {
            int64_t v[RB][CPL];
#pragma unroll
            for (int i = 0; i < RB; ++i) {
                const int u = runs ? __ffsll((long long)runs) - 1 : -1;
                runs &= runs - 1;
#pragma unroll
                for (int k = 0; k < CPL; ++k) v[i][k] = u >= 0 ? (int64_t)get64(sc.S + (base + u) * D + lane + 64 * k) : 0;
            }
#pragma unroll
            for (int i = 0; i < RB; ++i)
#pragma unroll
                for (int k = 0; k < CPL; ++k) acc[k] += v[i][k];
        }
        const int64_t orow = ((int64_t)b * g.n_q + kvh * G + h) * D;
        const Recip rc = reciprocal(l);
        int64_t amax = 0, over = 0;
#pragma unroll
        for (int k = 0; k < CPL; ++k) {
            if (acc[k] < ACC_LO || acc[k] > ACC_HI) {
                ++over;
                acc[k] = acc[k] < ACC_LO ? ACC_LO : ACC_HI;
            }
            out[orow + lane + 64 * k] = (int32_t)(wmul(acc[k], rc.r) >> rc.shift);
            amax = OpMax64::f(amax, acc[k] < 0 ? -acc[k] : acc[k]);
        }
        amax = wave_max_i64(amax);
        over = wave_sum_i64(over);
        if (lane == 0) {
            atomicMax(&S.macc, (unsigned long long)amax);
            if (over) atomicAdd(&S.aovf, (unsigned long long)over);
        }
    }
    __syncthreads();
    // (the serial path's rows lie over the sums)
    const uint32_t bad = S.bad;
    for (int h = wv; h < G; h += W)
        if (bad >> h & 1)
            serial_head<CPL, L::RS>(g, tabs, tabs->kc, tabs->vc, sc.qr + (crow + h) * D, b, kvh, T, 1, true, S.u.fb[wv],
                                    out + ((int64_t)b * g.n_q + kvh * G + h) * D, st);
    if (tid == 0) {
        if ((unsigned long long)T > st->n_tokens) atomicMax(&st->n_tokens, (unsigned long long)T);
        if (S.macc > st->max_abs_acc) atomicMax(&st->max_abs_acc, S.macc);
        if (S.aovf) atomicAdd(&st->acc_overflows, S.aovf);
        if (bad) atomicAdd(&st->serial_fallbacks, (unsigned long long)__popc(bad));
    }
}

template <int D, int KB, int NC, int NS>
hipError_t launch(hipStream_t s, const Geom &g, const Tables *t, const int32_t *q, int32_t *out, const int64_t *len,
                  const Scratch &sc, int r, int ub, int64_t nblk, const StepIn *step, LaunchEv ev,
                  DevStats *st) {
    const int64_t chains = (int64_t)g.batch * g.n_kv;
    const dim3 g1((unsigned)(chains * ((nblk + 4 * r - 1) / (4 * r)))), g2((unsigned)(chains * ((nblk + 4 * ub - 1) / (4 * ub))));
    if (step)
        hipExtLaunchKernelGGL((score_max_kernel<D, KB, NS, true>), g1, dim3(W * 64), 0, s, ev.start, nullptr, 0, g, t, q,
                              len, sc, r, st, *step);
    else
        hipExtLaunchKernelGGL((score_max_kernel<D, KB, NS, false>), g1, dim3(W * 64), 0, s, ev.start, nullptr, 0, g, t, q,
                              len, sc, r, st, StepIn{});
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipExtLaunchKernelGGL((sum_kernel<D, KB, NC, NS>), g2, dim3(W * 64), 0, s, nullptr, ev.stop, 0, g, t, out,
                          step ? (const int64_t *)step->len_out : len, sc, r, ub, st);
    return hipGetLastError();
}

// The scratch for a capacity, carved from p (null: only its size).
size_t carve(const Geom &g, int64_t capacity, uint8_t *p, Scratch *sc, size_t *front) {
    size_t o = 0;
    auto take = [&](size_t n) {
        uint8_t *a = p ? p + o : nullptr;
        o += (n + 255) / 256 * 256;
        return a;
    };
    const size_t chains = (size_t)g.batch * g.n_kv, gp = g.G > 4 ? 8 : 4;
    const int64_t nblk = (capacity + BT - 1) / BT;
    const int64_t nwg = (nblk + W - 1) / W < MAXWG ? (nblk + W - 1) / W : MAXWG;
    Scratch c{};
    c.nblk = (int32_t)nblk;
    c.nwg = (int32_t)nwg;
    c.done = (uint32_t *)take(chains * 4);
    if (front) *front = o;
    c.qbad = (uint32_t *)take(chains * 4);
    c.qr = (int32_t *)take(chains * gp * g.d * 4);
    c.bm = (int64_t *)take(chains * gp * c.nblk * 8);
    c.cm = (int64_t *)take(chains * gp * ((c.nblk + 3) / 4) * 8);
    c.meta = (uint64_t *)take(chains * gp * c.nwg * 8);
    c.S = (int64_t *)take(chains * gp * c.nwg * g.d * 8);
    if (sc) *sc = c;
    return o;
}

}  // namespace sp

// (A term t = floor(v_norm p c / 2^23) is at most 128 |c|; its digits are read from the fp64 sum while
// that stays below 2^29, i.e. t + 0x808080 below 2^27. Wider value centroids take the chunked attend.)
bool split_supported(const Geom &g, const Tables &th, int64_t capacity) {
    int64_t vmax = 0;
    for (int i = 0; i < (1 << g.vb); ++i) vmax = std::max<int64_t>(vmax, std::llabs(th.vc[i]));
    return 128 * vmax + 0x808080 < (int64_t(1) << 27) && (g.d == 64 || g.d == 128) && g.kb >= 2 && g.kb <= 4 && g.vb >= 1 && g.vb <= 3 && g.norm_frac == 9 &&
           g.G >= 1 && g.G <= 8 && g.kv_shift == 0 && g.gq == 0 &&
           capacity <= (int64_t)sp::MAXWG * sp::W * sp::MAXU * sp::BT;
}

size_t split_scratch_bytes(const Geom &g, int64_t capacity) { return sp::carve(g, capacity, nullptr, nullptr, nullptr); }

hipError_t launch_attend_split(hipStream_t s, const Geom &g, const Tables *t, const int32_t *q, int32_t *out,
                               const int64_t *len, ChunkScratch &cs, int64_t longest, const StepIn *step, LaunchEv ev,
                               DevStats *st) {
    using namespace sp;
    Scratch sc;
    size_t front = 0;
    if (carve(g, g.capacity, (uint8_t *)cs.p, &sc, &front) > cs.bytes || longest > g.capacity) return hipErrorInvalidValue;
    const hipError_t e = scratch_layout(s, cs, 0x53504C4954ull, front);
    if (e != hipSuccess) return e;
    const int64_t chains = (int64_t)g.batch * g.n_kv, nblk = longest > BT ? (longest + BT - 1) / BT : 1;
    auto clamp = [](int64_t v, int64_t lo, int64_t hi) { return v < lo ? lo : v > hi ? hi : v; };
    // blocks a wave scores, and blocks a unit: enough waves to fill the chip, then fewer, longer ones
    int r = 1;                                         // (a power of two: MAXU is a multiple)
    while (2 * r <= MAXU && chains * nblk >= 8192 * 2 * r) r *= 2;
    // (the waves of sum_kernel that the chip holds at once, by the registers each takes)
    const bool small = g.vb <= 2 && g.G <= 4;
    const int64_t resident = 256 * W * (g.d == 64 ? (small ? 4 : 3) : (small ? 3 : 2));
    int64_t ub = clamp((chains * nblk + resident - 1) / resident, 1, MAXU);
    const int64_t least = (nblk + MAXWG * W - 1) / (MAXWG * W);
    if (ub < least) ub = least;
    ub = clamp((ub + r - 1) / r * r, r, MAXU / r * r);
    const int nc = g.vb <= 2 ? 4 : 8, ns = g.G > 4 ? 2 : 1;
#define INSITU_SPLIT_CASE(DD, KK, CC, SS)                                                               \
    if (g.d == DD && g.kb == KK && nc == CC && ns == SS)                                                \
        return launch<DD, KK, CC, SS>(s, g, t, q, out, len, sc, r, (int)ub, nblk, step, ev, st);
#define INSITU_SPLIT_KB(DD, KK)                                                                          \
    INSITU_SPLIT_CASE(DD, KK, 4, 1) INSITU_SPLIT_CASE(DD, KK, 4, 2) INSITU_SPLIT_CASE(DD, KK, 8, 1)       \
    INSITU_SPLIT_CASE(DD, KK, 8, 2)
    INSITU_SPLIT_KB(64, 2)
    INSITU_SPLIT_KB(64, 3)
    INSITU_SPLIT_KB(64, 4)
    INSITU_SPLIT_KB(128, 2)
    INSITU_SPLIT_KB(128, 3)
    INSITU_SPLIT_KB(128, 4)
#undef INSITU_SPLIT_KB
#undef INSITU_SPLIT_CASE
    return hipErrorInvalidValue;
}

}  // namespace insitu
