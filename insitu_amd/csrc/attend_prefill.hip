// The prefill attend on matrix cores: attend_online_batch / attend_causal_batch
// (ops/attention.py:517-871), every query of a prompt over the rows before it, bit-exact
// with the sequential reference.
//
// A wave owns 16 rows, a row being one (query, query head) of a KV head's group, and
// walks the sequence's tokens in order, 16 at a time, as the reference does: it holds each
// row's running maximum, accumulator and denominator in registers, so no other workgroup is
// waited for and nothing is published or replayed. A workgroup's waves share one KV head's
// tokens, which they expand together into matrix operands in LDS, double-buffered.
//
// Scores. dot = sum_ch q[ch] * c[code_ch] exactly: q and the key centroids in three balanced signed
// bytes each, v_mfma_i32_16x16x64_i8 over the channels for every pair of digits, the products of
// equal weight in one int32 accumulator that carries into the next lower weight's: dot = 2^16 H + L.
// floor(dot k_norm / 2^24) is then int64 arithmetic, and the scores int32. Where that does not do (a
// value of q that needs its fourth byte, ||q||_1 max|c| from 2^46 on, a product past 2^55, which one
// bound a stage excludes or else the products are looked at, or a value term past three digits) the
// workgroup starts again with four digits and int64 scores (WIDE), which cover everything the
// reference computes: an int64 shifted right by 24 never reaches the 48-bit clamp, so that no score
// of this kernel overflows. A row with ||q||_1 max|c| from 2^51 on goes to the serial path.
//
// The matrix product's result has lane = (row, 4 tokens): the running maximum, the exp LUT and
// the terms floor(v_norm p c_v / 2^23) for every value code are computed there, and the terms'
// bytes (three balanced digits of the fp64 sum's mantissa) are at once the second product's
// operand: sum over (token, code) of [code of the token's channel] * term, with the one-hot
// codes staged in LDS. Its result has lane = (row, 4 channels a tile): the same row, so the
// rescale factor of an event is in the right lane too.
//
// Events (s > running maximum). A tile without one, the common case, only adds. Otherwise the
// tile's tokens fall into segments, one more than the row's events; the terms are masked by
// segment, and between two of them acc = floor(acc f / 2^15), l = floor(l f / 2^15).
//
// The per-token int32 clamp of acc (attention.py:502-503) cannot fire while |acc| plus the
// largest terms of all tokens since stays below 2^31 (a rescale never grows |acc|): one sum a
// wave proves it, refreshed from the accumulators when it gets large; a row where it cannot be
// proven is recomputed on the serial path (serial_head.h), as is one whose scores are not exact.
//
// What bounds it (SQ counters): VALU issue. A 4,096-token prompt takes a wave
// some 330 VALU and 25 matrix instructions a 16 x 16 tile, its share of the staging and its events
// included; they fill 62 % and 19 % of the SIMDs' cycles. 28 % of its tiles hold events (a count of
// random rows drawn as the benchmark's). A short prompt, two waves a SIMD or one, is bound by the
// longest walk's own latency: 0.1 us a row at d = 64, 0.1 a row and pass at d = 128. One accumulator
// instead of one a digit costs two VALU instructions a register and tile and frees 32 registers at
// d = 64 (64 at 128); the walk still spills some: 46 registers online and 42 two-pass at the 168 of three
// workgroups a CU, 26 to 62 at d = 128's 256.
// Measured (the kernel, Llama-3.2-1B shape, queries scaled as a model's): 4,096 tokens 883 us (the
// call 8,632 on the virtual batch of decode attends before); 333 tokens behind 2,000 219 us (797);
// 1,000 tokens at d = 128, 3b/3b, two-pass 201 us (1,923).
#include <type_traits>

#include "digits.h"
#include "query.h"
#include "serial_head.h"
#include "wave.h"

namespace insitu {
namespace pf {

// |dot k_norm| below this: floor(dot k_norm / 2^24) is above INT32_MIN, the narrow scores' "none yet"
constexpr double NARROW_LIMIT = 36028797018963968.0 - 16777216.0;
constexpr uint32_t LUT_N = LUT_SPAN + 1;               // p by floor index, the last entry 0
constexpr double TERM_MAGIC = 402653184.0 + 8421504.0; // 1.5 * 2^28 + 0x808080: ulp 2^-24
constexpr double TERM_LIMIT = 8355711.0;               // 0x7F7F7F: three balanced bytes
constexpr float ACC_BOUND = 2147483520.0f;             // the largest float below 2^31

// 16 bytes of a 4-byte aligned address: query rows, outputs and narrow planes
struct __attribute__((aligned(4))) u128 {
    uint32_t x, y, z, w;
};

enum Pass { MAXONLY = 0, FIXEDMAX = 1, ONLINE = 2 };

// Bytes b of four words, as the four dwords of bytes 0, 1, 2, 3.
__device__ __forceinline__ void bytes4(const uint32_t (&z)[4], uint32_t (&o)[4]) {
    const uint32_t a = perm(z[1], z[0], 0x05010400u), b = perm(z[3], z[2], 0x05010400u);
    const uint32_t c = perm(z[1], z[0], 0x07030602u), d = perm(z[3], z[2], 0x07030602u);
    o[0] = perm(b, a, 0x05040100u);
    o[1] = perm(b, a, 0x07060302u);
    o[2] = perm(d, c, 0x05040100u);
    o[3] = perm(d, c, 0x07060302u);
}
template <class S>
__device__ __forceinline__ S shfl_s(S v, int lane) {
    if constexpr (sizeof(S) == 8) {
        const uint32_t lo = (uint32_t)__shfl((int)(uint32_t)v, lane), hi = (uint32_t)__shfl((int)(uint32_t)((uint64_t)v >> 32), lane);
        return (S)(((uint64_t)hi << 32) | lo);
    } else {
        return (S)__shfl((int)v, lane);
    }
}

template <class S>
__device__ __forceinline__ S rdlane(S v, int lane) {   // lane wave-uniform
    if constexpr (sizeof(S) == 8)
        return (S)readlane64((int64_t)v, lane);
    else
        return (S)__builtin_amdgcn_readlane((int)v, lane);
}

// D: head dimension; NC: value code slots (4: up to 2-bit values, 8: 3-bit); W: waves; ST: tokens
// a stage.
template <int D, int NC, int W, int ST_>
struct Shape {
    static constexpr int ST = ST_;
    static constexpr int NT = ST / 16;                 // 16-token tiles of it
    static constexpr int KBLK = D / 64;                // 64-channel blocks of a score
    static constexpr int CT = D / 16;                  // 16-channel tiles of the accumulator
    static constexpr int PVK = NC / 4;                 // 64-deep blocks of (token, code) a tile
    static constexpr int RW = D == 64 ? 17 : 31;       // raw row stride, words (odd: no bank conflict)
    static constexpr int RS = D == 64 ? 60 : 116;      // widest row, bytes (4-bit keys, 3-bit values)
    static constexpr int THREADS = W * 64;
    static constexpr int UNITS = (ST * 8 + THREADS - 1) / THREADS;   // plane loads a thread (<= 8 planes)
};

template <int D, int NC, int W, int ST>
struct Lds {
    using C = Shape<D, NC, W, ST>;
    struct Op {
        v4i ka[2][C::NT][3][C::KBLK][64];              // key centroid digits: lane = (token, 16 channels)
        v4i oh[2][C::NT][C::PVK][C::CT][64];           // one-hot value codes: lane = (channel, tokens)
    };
    union {
        Op op;
        SerialLds<C::RS> fb[W];
    } u;
    uint32_t raw[2][C::ST][C::RW];
    alignas(16) int32_t kn[2][C::ST], vn[2][C::ST];
    int32_t knmax[2], vnmax[2];
    alignas(16) uint32_t dig[3][4];                    // 16 centroids' digits, a byte each
    uint16_t lut[LUT_N + 7];
    int rerun;
    unsigned long long events, rerr, fallbacks, mabs, macc;
};

// A workgroup's walk over its tokens, and its rows' outputs. Narrow scores: returns true when
// they did not do (workgroup-uniform; nothing is written then). WIDE: int64 scores and a fourth
// digit of q.
template <int D, int NC, int W, int ST, bool TWO_PASS, bool WIDE>
__device__ __forceinline__ bool prefill_rows(const Geom &g, const Tables *__restrict__ tabs,
                                             const int32_t *__restrict__ q, int32_t *out, int64_t base, int64_t n_q,
                                             DevStats *st, Lds<D, NC, W, ST> &S) {
    using C = Shape<D, NC, W, ST>;
    using SC = typename std::conditional<WIDE, int64_t, int32_t>::type;
    constexpr int NQ = WIDE ? 4 : 3;                   // digits of q
    constexpr SC LO = WIDE ? (SC)SCORE_LO : (SC)INT32_MIN;
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 15, grp = lane >> 4;
    const int G = g.G;
    // the longest contexts first; a KV head's workgroups a multiple of n_kv apart
    const int64_t rows = n_q * G;
    const int64_t nblk = (rows + W * 16 - 1) / (W * 16);
    const int64_t blk = nblk - 1 - (int64_t)(blockIdx.x / (unsigned)g.n_kv);
    const int kvh = (int)(blockIdx.x % (unsigned)g.n_kv);
    const uint8_t *hb = plane_ptr(g, 0, kvh, 0);
    const int64_t row0 = (blk * W + wv) * 16;          // this wave's first row
    const int64_t t_all = base + n_q;                  // rows the sequence holds for the last query
    const int64_t last_row = (blk + 1) * (W * 16) < rows ? (blk + 1) * (W * 16) - 1 : rows - 1;
    const int64_t tmax = base + last_row / G + 1;      // the workgroup's longest context

    // -- tables, and each row's query digits -------------------------------------------------
    if (tid == 0) {
        // (not in the wide walk: a wave of this workgroup may still be about to read it there)
        if constexpr (!WIDE) S.rerun = 0;
        S.events = S.rerr = S.fallbacks = S.mabs = S.macc = 0;
    }
    const int kb = g.kb, vb = g.vb;
    if (tid < 256) {
        const int32_t x = tabs->exp_table[tid];
        const int32_t kc = tid < (1 << kb) ? (int32_t)tabs->kc[tid] : 0;
#pragma unroll
        for (int i = 0; i < LUT_SPAN / 256; ++i) S.lut[256 * i + tid] = (uint16_t)(x >> i);
        if (tid == 0) S.lut[LUT_SPAN] = 0;
        if (tid < 16) {
            const uint32_t z = balanced(kc);   // |c| < 2^20
#pragma unroll
            for (int l = 0; l < 3; ++l) ((uint8_t *)S.dig[l])[tid] = (uint8_t)(z >> (8 * l));
        }
    }
    double vcs[NC];                                    // value centroids / 2^23
    double vcmax = 0.0;
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        vcs[i] = __longlong_as_double(uni64(__double_as_longlong(i < (1 << vb) ? (double)tabs->vc[i] * 0x1p-23 : 0.0)));
        vcmax = fmax(vcmax, fabs(vcs[i]));
    }
    const uint32_t delta_max = (uint32_t)tabs->delta_max;

    // this lane's row and the digits of 16 of its channels a block
    const bool valid = row0 + col < rows;
    const int64_t rowc = valid ? row0 + col : rows - 1;
    const int32_t limit = (int32_t)(base + rowc / G + 1);      // the row's context length
    bool bad;                                          // its arithmetic is not proven: serial path
    double bq;                                         // largest ||q||_1 max|c| of the wave's rows
    bool over = false;                                 // narrow scores: a value too large
    v4i qd[NQ][C::KBLK];
    {
        const int32_t *qp = q + ((rowc / G) * g.n_q + (int64_t)kvh * G + rowc % G) * D + grp * 16;
        unsigned long long rerr = 0;
        uint32_t any3 = 0, big = 0;
        int64_t l1 = 0;
#pragma unroll
        for (int b = 0; b < C::KBLK; ++b) {
            uint32_t z[16];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const u128 v = valid ? *(const u128 *)(qp + b * 64 + 4 * i) : u128{0, 0, 0, 0};
                const int32_t x[4] = {(int32_t)v.x, (int32_t)v.y, (int32_t)v.z, (int32_t)v.w};
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const uint32_t ax = x[j] < 0 ? 0u - (uint32_t)x[j] : (uint32_t)x[j];
                    l1 += ax;
                    rerr += ax >= (uint32_t)Q_ROT_LIMIT ? 1 : 0;
                    big |= ax >> 30;
                    z[4 * i + j] = balanced(x[j]);
                }
            }
            // byte k of the 16: channel k, or with 4-bit keys the even and the odd channels of 8
            // in turn (the order the nibbles come in)
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const int e = 8 * (w >> 1) + (w & 1);
                uint32_t zz[4], o[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) zz[i] = kb == 4 ? z[e + 2 * i] : z[4 * w + i];
                bytes4(zz, o);
#pragma unroll
                for (int i = 0; i < NQ; ++i) qd[i][b][w] = (int)o[i];
                any3 |= o[3];
            }
        }
        l1 += shfl_s<int64_t>(l1, lane ^ 16);
        l1 += shfl_s<int64_t>(l1, lane ^ 32);
        big |= (uint32_t)__shfl((int)big, lane ^ 16);
        big |= (uint32_t)__shfl((int)big, lane ^ 32);
        const double b1 = (double)l1 * tabs->kc_absmax;
        bad = !(b1 < DOT_LIMIT) || big != 0;           // its scores may not be exact
        bq = bad ? 0.0 : b1;
        if (!WIDE && (any3 != 0 || !(bq < 0x1p46))) over = true;   // a fourth digit; |dot| / 2^16 near 2^31
        __syncthreads();                               // the counters' zeros
        if (rerr) atomicAdd(&S.rerr, rerr);
#pragma unroll
        for (int o = 1; o < 16; o <<= 1) bq = fmax(bq, __shfl_xor(bq, o));
    }
    const int32_t wmin = (int32_t)(base + (row0 < rows ? row0 : rows - 1) / G + 1);       // the wave's contexts
    const int32_t wmax = row0 < rows ? (int32_t)(base + ((row0 + 16 < rows ? row0 + 16 : rows) - 1) / G + 1) : 0;

    // -- staging -------------------------------------------------------------------------
    // Plane p of the stage's tokens, 16 bytes a load (a narrower record's tail is the next ones',
    // or the span's padding: a span holds 16 bytes a token).
    u128 rg[C::UNITS];
    const uint8_t *src[C::UNITS];
    int width[C::UNITS];
    uint32_t *dst[C::UNITS];
#pragma unroll
    for (int u = 0; u < C::UNITS; ++u) {
        const int unit = tid + u * C::THREADS, p = C::ST == 64 ? uni32(unit / C::ST) : unit / C::ST;
        const bool in = p < g.n_planes;
        width[u] = in ? g.plane_w[p] : 0;
        src[u] = hb + (in ? (int64_t)p * g.span : 0);
        dst[u] = &S.raw[0][unit % C::ST][in ? g.plane_lo[p] / 4 : 0];
    }
    auto load_raw = [&](int s) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < C::UNITS; ++u) {
            const int t = s * C::ST + (tid + u * C::THREADS) % C::ST;
            if (width[u]) rg[u] = *(const u128 *)(src[u] + (int64_t)((t < (int)t_all ? t : (int)t_all - 1) * width[u]));
        }
    };
    auto store_raw = [&](int rb) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < C::UNITS; ++u) {
            uint32_t *d = dst[u] + rb * (C::ST * C::RW);
            if (width[u] >= 4) d[0] = rg[u].x;
            if (width[u] >= 8) d[1] = rg[u].y;
            if (width[u] == 16) {
                d[2] = rg[u].z;
                d[3] = rg[u].w;
            }
        }
    };
    // raw rows -> matrix operands
    auto expand = [&](int bf, bool values) __attribute__((always_inline)) {
        const uint4 d0 = *(const uint4 *)S.dig[0], d1 = *(const uint4 *)S.dig[1], d2 = *(const uint4 *)S.dig[2];
        const uint32_t dg[3][4] = {{d0.x, d0.y, d0.z, d0.w}, {d1.x, d1.y, d1.z, d1.w}, {d2.x, d2.y, d2.z, d2.w}};
#pragma unroll
        for (int j = 0; j < (C::ST * (D / 16) + C::THREADS - 1) / C::THREADS; ++j) {
            const int u = tid + j * C::THREADS;
            if (C::ST * (D / 16) % C::THREADS && u >= C::ST * (D / 16)) break;
            const int tok = u % C::ST, b = u / C::ST;
            const int off = b * 16 * kb, wd = off >> 5, sh = off & 31;
            const uint32_t lo = S.raw[bf][tok][wd], hi = S.raw[bf][tok][wd + 1];
            const uint64_t x = (((uint64_t)hi << 32) | lo) >> sh;
            v4i o[3];
            if (kb == 4)
                expand16<4>(x, dg, o);
            else if (kb == 3)
                expand16<3>(x, dg, o);
            else
                expand16<2>(x, dg, o);
#pragma unroll
            for (int l = 0; l < 3; ++l) S.u.op.ka[bf][tok >> 4][l][b >> 2][(b & 3) * 16 + (tok & 15)] = o[l];
        }
        if (values) {
            const int kw = g.key_bytes / 4;
#pragma unroll
            for (int j = 0; j < C::NT * 4 * D / C::THREADS; ++j) {
                const int u = tid + j * C::THREADS;
                const int ch = u % D, tg = u / D;
                const int bit = ch * vb, wd = kw + (bit >> 5), sh = bit & 31;
                uint32_t code[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t *rp = &S.raw[bf][4 * tg + i][wd];
                    const uint32_t x = NC == 4 ? rp[0] >> sh : __builtin_amdgcn_alignbit(rp[1], rp[0], sh);
                    code[i] = x & ((1u << vb) - 1u);
                }
                if constexpr (NC == 4) {
                    v4i o;
#pragma unroll
                    for (int i = 0; i < 4; ++i) o[i] = (int)(1u << (8 * code[i]));
                    S.u.op.oh[bf][tg >> 2][0][ch >> 4][(tg & 3) * 16 + (ch & 15)] = o;
                } else {
#pragma unroll
                    for (int k = 0; k < 2; ++k) {
                        v4i o;
#pragma unroll
                        for (int i = 0; i < 2; ++i) {
                            const uint64_t h = 1ull << (8 * code[2 * k + i]);
                            o[2 * i] = (int)(uint32_t)h;
                            o[2 * i + 1] = (int)(uint32_t)(h >> 32);
                        }
                        S.u.op.oh[bf][tg >> 2][k][ch >> 4][(tg & 3) * 16 + (ch & 15)] = o;
                    }
                }
            }
        }
        if (wv == W - 1) {
            const int tok = lane % C::ST;
            const uint32_t nw = S.raw[bf][tok][g.row_bytes / 4 - 1];
            const int32_t kn = (int16_t)(uint16_t)nw, vn = (int16_t)(uint16_t)(nw >> 16);
            if (lane < C::ST) {
                S.kn[bf][tok] = kn;
                S.vn[bf][tok] = vn;
            }
            const int32_t km = wave_max_i32(kn < 0 ? -kn : kn), vm = wave_max_i32(vn < 0 ? -vn : vn);
            if (lane == 0) {
                S.knmax[bf] = km;
                S.vnmax[bf] = vm;
            }
        }
    };

    // -- the walk ------------------------------------------------------------------------
    SC m = LO, smin = 0;
    v4i acc[C::CT];                                    // lane = (row, 4 channels of each tile)
    uint32_t lp = 0;                                   // this lane's part of the denominator since the last event or fold
    uint64_t l64 = 0;                                  // the row's denominator up to there
    uint32_t n_events = 0;
    float bsum = 0.0f;                                 // bound of |acc| over the wave's rows
#pragma unroll
    for (int c = 0; c < C::CT; ++c) acc[c] = v4i{0, 0, 0, 0};

    auto row_acc_max = [&]() __attribute__((always_inline)) -> double {
        uint32_t mx = 0;
#pragma unroll
        for (int c = 0; c < C::CT; ++c)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int32_t a = acc[c][i];
                const uint32_t aa = a < 0 ? 0u - (uint32_t)a : (uint32_t)a;
                mx = aa > mx ? aa : mx;
            }
        uint32_t o = (uint32_t)__shfl((int)mx, lane ^ 16);
        mx = o > mx ? o : mx;
        o = (uint32_t)__shfl((int)mx, lane ^ 32);
        return (double)(o > mx ? o : mx);
    };
    auto lut = [&](uint32_t d) __attribute__((always_inline)) -> uint32_t {
        // floor(d * log2e / 2^24), at most LUT_SPAN (d <= delta_max)
        return S.lut[__umulhi(d, (uint32_t)LOG2E_Q16 << 8)];
    };
    // a distance, at most delta_max
    auto clip = [&](SC hi, SC lo) __attribute__((always_inline)) -> uint32_t {
        if constexpr (WIDE) {
            return hi - lo < (SC)delta_max ? (uint32_t)(hi - lo) : delta_max;
        } else {
            const uint32_t w = (uint32_t)hi - (uint32_t)lo;
            return w < delta_max ? w : delta_max;
        }
    };

    // the row's denominator, in its four lanes
    auto denominator = [&]() __attribute__((always_inline)) -> uint64_t {
        uint64_t tot = lp;
        tot += shfl_s<uint64_t>(tot, lane ^ 16);
        tot += shfl_s<uint64_t>(tot, lane ^ 32);
        return l64 + tot;
    };

    // acc += the terms in A: the sums of the highest digits first, each carried into the next
    // product's accumulator. WIDE's terms have a fourth digit, of weight 2^21.
    auto accumulate = [&](const v4i (&A)[WIDE ? 4 : 3][C::PVK], int bf, int tl) __attribute__((always_inline)) {
        constexpr int GC = 4;                          // channel tiles at a time, to cover the products' latency
#pragma unroll
        for (int c0 = 0; c0 < C::CT; c0 += GC) {
            v4i o[GC][C::PVK], t[GC];
#pragma unroll
            for (int c = 0; c < GC; ++c)
#pragma unroll
                for (int k = 0; k < C::PVK; ++k) o[c][k] = S.u.op.oh[bf][tl][k][c0 + c][lane];
#pragma unroll
            for (int c = 0; c < GC; ++c) {
                t[c] = v4i{0, 0, 0, 0};
#pragma unroll
                for (int k = 0; k < C::PVK; ++k) {
                    t[c] = mma(o[c][k], A[2][k], t[c]);
                    if constexpr (WIDE) t[c] = mma(o[c][k] << 5, A[3][k], t[c]);
                }
            }
#pragma unroll
            for (int c = 0; c < GC; ++c) {
                t[c] = t[c] << 8;
#pragma unroll
                for (int k = 0; k < C::PVK; ++k) t[c] = mma(o[c][k], A[1][k], t[c]);
            }
#pragma unroll
            for (int c = 0; c < GC; ++c) {
                t[c] = (t[c] << 8) + acc[c0 + c];
#pragma unroll
                for (int k = 0; k < C::PVK; ++k) t[c] = mma(o[c][k], A[0][k], t[c]);
                acc[c0 + c] = t[c];
            }
        }
    };

    // one 16-token tile of the stage in buffer bf; t0 its first token. diag: some rows' contexts
    // may end in it. check: look at the products; tight: prove the clamp row by row.
    auto tile = [&](auto passc, int bf, int tl, int32_t t0, bool diag, bool check, bool tight) __attribute__((always_inline)) {
        constexpr Pass P = decltype(passc)::value;
        SC s[4];
        if constexpr (!WIDE) {
            // dot = 2^16 H + L, each digit weight's sum carried into the next product's accumulator
            // (|H| < 2^31, so what wraps on the way comes back)
            v4i a[C::KBLK][3], H = {0, 0, 0, 0}, L = {0, 0, 0, 0};
#pragma unroll
            for (int b = 0; b < C::KBLK; ++b)
#pragma unroll
                for (int l = 0; l < 3; ++l) a[b][l] = S.u.op.ka[bf][tl][l][b][lane];
#pragma unroll
            for (int k = 4; k >= 2; --k) {
                if (k < 4) H = H << 8;
#pragma unroll
                for (int b = 0; b < C::KBLK; ++b)
#pragma unroll
                    for (int l = 0; l < 3; ++l)
                        if (k - l >= 0 && k - l < 3) H = mma(a[b][l], qd[k - l][b], H);
            }
#pragma unroll
            for (int k = 1; k >= 0; --k) {
                if (k < 1) L = L << 8;
#pragma unroll
                for (int b = 0; b < C::KBLK; ++b)
#pragma unroll
                    for (int l = 0; l <= k; ++l) L = mma(a[b][l], qd[k - l][b], L);
            }
            const int4 k4 = *(const int4 *)&S.kn[bf][tl * 16 + grp * 4];
            const int32_t kn[4] = {k4.x, k4.y, k4.z, k4.w};
            int64_t x[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                x[i] = (int64_t)H[i] * kn[i] + (((int64_t)L[i] * kn[i]) >> 16);    // floor(dot k_norm / 2^16)
                s[i] = (int32_t)(uint32_t)((uint64_t)x[i] >> 8);
            }
            if (check) {
#pragma unroll
                for (int i = 0; i < 4; ++i) over |= ((x[i] >> 8) != (int64_t)s[i] || s[i] == LO) && !bad;
            }
        } else {
            v4i T[NQ + 2];
#pragma unroll
            for (int k = 0; k < NQ + 2; ++k) T[k] = v4i{0, 0, 0, 0};
#pragma unroll
            for (int b = 0; b < C::KBLK; ++b) {
                v4i a[3];
#pragma unroll
                for (int l = 0; l < 3; ++l) a[l] = S.u.op.ka[bf][tl][l][b][lane];
#pragma unroll
                for (int l = 0; l < 3; ++l)
#pragma unroll
                    for (int i = 0; i < NQ; ++i) T[l + i] = mma(a[l], qd[i][b], T[l + i]);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                int64_t dot = 0;
#pragma unroll
                for (int k = NQ + 1; k >= 0; --k) dot = wadd(wmul(dot, 256), T[k][i]);
                s[i] = wmul(dot, S.kn[bf][tl * 16 + grp * 4 + i]) >> (CENT_FRAC + 9);
            }
        }
        const int32_t tg = t0 + grp * 4;               // this lane's first token
        if (diag) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const bool in = tg + i < limit;
                if (P != FIXEDMAX) smin = in && s[i] < smin ? s[i] : smin;
                s[i] = in ? s[i] : LO;
            }
        } else if (P != FIXEDMAX) {
#pragma unroll
            for (int i = 0; i < 4; ++i) smin = s[i] < smin ? s[i] : smin;
        }
        const SC s01 = s[0] > s[1] ? s[0] : s[1], s23 = s[2] > s[3] ? s[2] : s[3];
        const SC mx = s01 > s23 ? s01 : s23;
        if constexpr (P == MAXONLY) {
            m = mx > m ? mx : m;                       // this lane's tokens; joined after the pass
            return;
        }
        // distances below the running maximum, then p, the terms of every (token, code) as digit
        // bytes. NC = 4: dword = token; NC = 8: block = token pair, dword = (token, half its codes)
        v4i A[WIDE ? 4 : 3][C::PVK];
        uint32_t p[4];
        auto terms = [&](bool mask, const uint32_t (&dl)[4]) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < 4; ++i) p[i] = lut(dl[i]);
            if (mask) {
#pragma unroll
                for (int i = 0; i < 4; ++i) p[i] = tg + i < limit ? p[i] : 0u;
            }
            const int4 vn4 = *(const int4 *)&S.vn[bf][tl * 16 + grp * 4];
            const int32_t w[4] = {__mul24(vn4.x, (int)p[0]), __mul24(vn4.y, (int)p[1]), __mul24(vn4.z, (int)p[2]),
                                  __mul24(vn4.w, (int)p[3])};
            if (P != MAXONLY && tight) {
                double sum = 4.0;
#pragma unroll
                for (int i = 0; i < 4; ++i) sum += fabs((double)w[i]) * vcmax;
                sum += __shfl_xor(sum, 16);
                sum += __shfl_xor(sum, 32);
                if (!(row_acc_max() + sum <= 2147483647.0)) bad = true;
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const double wd = (double)w[i];
#pragma unroll
                for (int k4 = 0; k4 < NC / 4; ++k4) {
                    const int kbk = NC == 4 ? 0 : i >> 1, dw = NC == 4 ? i : 2 * (i & 1) + k4;
                    if constexpr (!WIDE) {
                        uint32_t yl[4], yh[4];
#pragma unroll
                        for (int k = 0; k < 4; ++k) {
                            const uint64_t y = (uint64_t)__double_as_longlong(fma(wd, vcs[4 * k4 + k], TERM_MAGIC));
                            yl[k] = (uint32_t)y;
                            yh[k] = (uint32_t)(y >> 32);
                        }
                        const uint32_t l01 = perm(yl[1], yl[0], 0x0C0C0703u), l23 = perm(yl[3], yl[2], 0x07030C0Cu);
                        const uint32_t h01 = perm(yh[1], yh[0], 0x05010400u), h23 = perm(yh[3], yh[2], 0x05010400u);
                        A[0][kbk][dw] = (int)((l01 | l23) ^ 0x80808080u);
                        A[1][kbk][dw] = (int)(perm(h23, h01, 0x05040100u) ^ 0x80808080u);
                        A[2][kbk][dw] = (int)(perm(h23, h01, 0x07060302u) ^ 0x80808080u);
                    } else {
                        uint32_t z[4], d2 = 0, d3 = 0;
#pragma unroll
                        for (int k = 0; k < 4; ++k) {
                            const int32_t t = (int32_t)floor(wd * vcs[4 * k4 + k]);   // |t| < 2^27: top at most 2^11
                            z[k] = ((uint32_t)t + 0x8080u) ^ 0x8080u;
                            const int32_t top = (int32_t)((uint32_t)t + 0x8080u) >> 16;
                            d2 |= (uint32_t)(top & 31) << (8 * k);
                            d3 |= ((uint32_t)(top >> 5) & 0xFFu) << (8 * k);
                        }
                        const uint32_t a = perm(z[1], z[0], 0x05010400u), b = perm(z[3], z[2], 0x05010400u);
                        A[0][kbk][dw] = (int)perm(b, a, 0x05040100u);
                        A[1][kbk][dw] = (int)perm(b, a, 0x07060302u);
                        A[2][kbk][dw] = (int)d2;
                        A[WIDE ? 3 : 0][kbk][dw] = (int)d3;
                    }
                }
                if (D == 128) __builtin_amdgcn_sched_barrier(0);     // few sums in flight: registers
            }
        };
        const bool plain = P != ONLINE || __ballot(mx > m) == 0;
        if (plain) {
            if constexpr (WIDE) {
                if (__ballot(m - mx < (SC)delta_max) == 0) return;
            } else {
                if (__ballot((uint32_t)m - (uint32_t)mx < delta_max) == 0) return;   // every p is 0
            }
        }
        if (P != ONLINE || (plain && !diag)) {
            const uint32_t dl[4] = {clip(m, s[0]), clip(m, s[1]), clip(m, s[2]), clip(m, s[3])};
            terms(P != ONLINE && diag, dl);
            lp += (p[0] + p[1]) + (p[2] + p[3]);
            accumulate(A, bf, tl);
            return;
        }
        if constexpr (P != ONLINE) return;
        // a tile with events, or at a row's end: its tokens in segments (bits 8 i of seg the segment
        // of token i)
        uint32_t dl[4], fe[4], seg = 0;
        SC e = m;                                      // the maximum before this lane's tokens
        const unsigned long long evl = __ballot(mx > m);
        const bool single = (evl & (evl - 1)) == 0;    // at most one lane holds events
        if (!single) {
            const SC a = shfl_s<SC>(mx, lane - 16), b = shfl_s<SC>(mx, lane - 32), c = shfl_s<SC>(mx, lane - 48);
            if (grp > 0) e = a > e ? a : e;
            if (grp > 1) e = b > e ? b : e;
            if (grp > 2) e = c > e ? c : e;
        } else if (evl) {                              // the row's later tokens see its maximum
            const int l = __ffsll((long long)evl) - 1;
            const SC t = rdlane<SC>(mx, l);
            if (col == (l & 15)) e = grp > (l >> 4) ? t : e;
        }
        uint32_t n = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const bool ev = s[i] > e;
            const uint32_t dd = clip(ev ? s[i] : e, ev ? e : s[i]);
            fe[i] = ev ? dd + 1u : 0u;                 // an event's distance, + 1
            dl[i] = ev ? 0u : dd;
            e = ev ? s[i] : e;
            n += ev ? 1 : 0;
            seg |= n << (8 * i);
        }
        int row_ev = 0;                                // the row's events
        if (!single) {
            const uint32_t n1 = (uint32_t)__shfl((int)n, lane - 16), n2 = (uint32_t)__shfl((int)n, lane - 32),
                           n3 = (uint32_t)__shfl((int)n, lane - 48);
            const uint32_t off = (grp > 0 ? n1 : 0) + (grp > 1 ? n2 : 0) + (grp > 2 ? n3 : 0);
            seg += off * 0x01010101u;                  // at most 16
            row_ev = __shfl((int)(off + n), 48 + col);
            m = shfl_s<SC>(e, 48 + col);
        } else if (evl) {
            const int l = __ffsll((long long)evl) - 1;
            const uint32_t nl = (uint32_t)__builtin_amdgcn_readlane((int)n, l);
            const SC t = rdlane<SC>(mx, l);
            if (col == (l & 15)) {
                if (grp > (l >> 4)) seg += nl * 0x01010101u;
                row_ev = (int)nl;
                m = t;
            }
        }
        n_events += n;
        terms(true, dl);
        for (int sg = 0;; ++sg) {
            v4i B[WIDE ? 4 : 3][C::PVK];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const bool in = ((seg >> (8 * i)) & 0xFFu) == (uint32_t)sg;
                lp += in ? p[i] : 0u;
#pragma unroll
                for (int l = 0; l < (WIDE ? 4 : 3); ++l) {
                    if constexpr (NC == 4) {
                        B[l][0][i] = in ? A[l][0][i] : 0;
                    } else {
                        B[l][i >> 1][2 * (i & 1)] = in ? A[l][i >> 1][2 * (i & 1)] : 0;
                        B[l][i >> 1][2 * (i & 1) + 1] = in ? A[l][i >> 1][2 * (i & 1) + 1] : 0;
                    }
                }
            }
            accumulate(B, bf, tl);
            const bool has = row_ev > sg;
            if (__ballot(has) == 0) break;
            // the event that opens segment sg + 1 of the row (rows without one: factor 1)
            uint32_t fd = 0;
#pragma unroll
            for (int i = 0; i < 4; ++i) fd = ((seg >> (8 * i)) & 0xFFu) == (uint32_t)(sg + 1) && fe[i] ? fe[i] : fd;
            if (single) {
                fd = (uint32_t)__builtin_amdgcn_readlane((int)fd, __ffsll((long long)evl) - 1);
            } else {
                fd |= (uint32_t)__shfl((int)fd, lane ^ 16);
                fd |= (uint32_t)__shfl((int)fd, lane ^ 32);
            }
            const int32_t f = has ? (int32_t)lut(fd - 1u) : 1 << PROB_FRAC;
#pragma unroll
            for (int c = 0; c < C::CT; ++c) {
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[c][i] = (int32_t)(((int64_t)acc[c][i] * f) >> PROB_FRAC);
                __builtin_amdgcn_sched_barrier(0);     // few products in flight: registers
            }
            const uint64_t l = denominator();
            if (has) {
                l64 = (l * (uint64_t)f) >> PROB_FRAC;
                lp = 0;
            }
        }
    };

    auto sweep = [&](auto passc) __attribute__((always_inline)) {
        constexpr Pass P = decltype(passc)::value;
        const int nst = (int)((tmax + C::ST - 1) / C::ST);
        load_raw(0);
        store_raw(0);
        __syncthreads();
        expand(0, P != MAXONLY);
        if (nst > 1) load_raw(1);
        for (int s = 0; s < nst; ++s) {
            const int bf = s & 1;
            if (s + 1 < nst) store_raw(bf ^ 1);
            if (s + 2 < nst) load_raw(s + 2);
            __syncthreads();
            if (s + 1 < nst) expand(bf ^ 1, P != MAXONLY);
            // narrow scores fit 32 bits when the largest product does (else they are looked at)
            const bool check = uni32(!(bq * (double)S.knmax[bf] < NARROW_LIMIT));
            // the largest |term| of the stage's tokens, p at most 1, and the floor
            const double term = (double)uni32(S.vnmax[bf]) * 32768.0 * vcmax + 2.0;
            if (!WIDE && term > TERM_LIMIT) over = true;
            bool tight = false;
            if (P != MAXONLY) {                        // the clamp certificate, a stage at a time
                const float add = (float)(term * C::ST) * 1.0000002f;
                bsum += add;
                if (uni32(!(bsum <= ACC_BOUND))) {
                    double mxr = bad ? 0.0 : row_acc_max();
#pragma unroll
                    for (int o = 1; o < 16; o <<= 1) mxr = fmax(mxr, __shfl_xor(mxr, o));
                    bsum = (float)mxr * 1.0000002f + add;
                    tight = uni32(!(bsum <= ACC_BOUND));
                }
            }
            const int32_t ts = s * C::ST;
            for (int tl = 0; tl < C::NT && ts + tl * 16 < wmax; ++tl)
                tile(passc, bf, tl, ts + tl * 16, ts + tl * 16 + 16 > wmin, check, tight);
            // a stage adds at most 16 tokens of 2^15 to a lane's 32 bits
            if (P != MAXONLY && (s & 4095) == 4095) {
                l64 = denominator();
                lp = 0;
            }
        }
        __syncthreads();
    };
    if constexpr (TWO_PASS) {
        sweep(std::integral_constant<Pass, MAXONLY>{});
        SC o = shfl_s<SC>(m, lane ^ 16);
        m = o > m ? o : m;
        o = shfl_s<SC>(m, lane ^ 32);
        m = o > m ? o : m;
        sweep(std::integral_constant<Pass, FIXEDMAX>{});
    } else {
        sweep(std::integral_constant<Pass, ONLINE>{});
    }
    if constexpr (!WIDE) {
        // From this barrier on nothing writes the flag, so that the whole workgroup takes the one way
        // or the other; the wide walk writes nothing before its first barrier that is read here.
        if (over && valid) S.rerun = 1;
        __syncthreads();
        if (S.rerun) return true;
    }

    // -- finalize --------------------------------------------------------------------------
    {
        const Recip rc = reciprocal((int64_t)denominator());
        const bool mine = valid && !bad;
        const int64_t at = ((rowc / G) * g.n_q + (int64_t)kvh * G + rowc % G) * D;
        int64_t macc = 0;
#pragma unroll
        for (int c = 0; c < C::CT; ++c) {
            uint32_t o[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int64_t a = acc[c][i], aa = a < 0 ? -a : a;
                macc = aa > macc ? aa : macc;
                o[i] = (uint32_t)(wmul(a, rc.r) >> rc.shift);
            }
            if (mine) *(u128 *)(out + at + c * 16 + grp * 4) = u128{o[0], o[1], o[2], o[3]};
        }
        const int64_t mp = (int64_t)m < 0 ? -(int64_t)m : (int64_t)m, mn = -(int64_t)smin;
        const int64_t ev = wave_sum_i64(mine ? n_events : 0);
        const int64_t ma = wave_max_i64(mine ? (mp > mn ? mp : mn) : 0), mc = wave_max_i64(mine ? macc : 0);
        if (lane == 0) {
            if (ev) atomicAdd(&S.events, (unsigned long long)ev);
            atomicMax(&S.mabs, (unsigned long long)ma);
            atomicMax(&S.macc, (unsigned long long)mc);
        }
    }
    // the rows whose arithmetic could not be proven: the reference loop
    const unsigned long long bads = __ballot(valid && bad) & 0xFFFFull;
    if (bads) {
        for (int c = 0; c < 16; ++c) {
            if (!(bads >> c & 1)) continue;
            const int64_t row = row0 + c, at = ((row / G) * g.n_q + (int64_t)kvh * G + row % G) * D;
            if (lane == 0) atomicAdd(&S.fallbacks, 1ull);
            serial_head<D / 64, C::RS>(g, tabs, tabs->kc, tabs->vc, q + at, 0, kvh, base + row / G + 1, TWO_PASS ? 1 : 0,
                                       true, S.u.fb[wv], out + at, st);
        }
    }
    __syncthreads();
    // one set of counters a workgroup (equal addresses apply one at a time); a maximum only when
    // it is one as far as this workgroup can see
    if (tid == 0) {
        if (S.events) atomicAdd(&st->rescale_events, S.events);
        if (S.rerr) atomicAdd(&st->range_errors, S.rerr);
        if (S.fallbacks) atomicAdd(&st->serial_fallbacks, S.fallbacks);
        if (S.mabs > st->max_abs_score) atomicMax(&st->max_abs_score, S.mabs);
        if (S.macc > st->max_abs_acc) atomicMax(&st->max_abs_acc, S.macc);
        if (blk == nblk - 1 && kvh == 0) atomicMax(&st->n_tokens, (unsigned long long)t_all);
    }
    return false;
}

// Not inlined, so that its registers are its own: it is entered when narrow scores did not do.
template <int D, int NC, int W, int ST, bool TWO_PASS>
__device__ __attribute__((noinline)) void prefill_rows_wide(const Geom *g, const Tables *tabs, const int32_t *q, int32_t *out,
                                                            int64_t base, int64_t n_q, DevStats *st, Lds<D, NC, W, ST> *S) {
    prefill_rows<D, NC, W, ST, TWO_PASS, true>(*g, tabs, q, out, base, n_q, st, *S);
}

template <int D, int NC, int W, int ST, bool TWO_PASS>
__global__ void __launch_bounds__(W * 64, D == 64 && ST == 32 && NC == 4 ? 3 : 2) prefill_kernel(Geom g, const Tables *__restrict__ tabs,
                                                           const int32_t *__restrict__ q, int32_t *out,
                                                           int64_t base, int64_t n_q, DevStats *st) {
    __shared__ Lds<D, NC, W, ST> S;
    if (prefill_rows<D, NC, W, ST, TWO_PASS, false>(g, tabs, q, out, base, n_q, st, S))
        prefill_rows_wide<D, NC, W, ST, TWO_PASS>(&g, tabs, q, out, base, n_q, st, &S);
}

template <int D, int NC, int W, int ST>
hipError_t launch(hipStream_t s, const Geom &g, const Tables *t, const int32_t *q, int32_t *out, int64_t base,
                  int64_t n_q, int two_pass, LaunchEv ev, DevStats *st) {
    const int64_t blocks = (n_q * g.G + W * 16 - 1) / (W * 16) * g.n_kv;
    if (two_pass)
        hipExtLaunchKernelGGL((prefill_kernel<D, NC, W, ST, true>), dim3((unsigned)blocks), dim3(W * 64), 0, s, ev.start,
                              ev.stop, 0, g, t, q, out, base, n_q, st);
    else
        hipExtLaunchKernelGGL((prefill_kernel<D, NC, W, ST, false>), dim3((unsigned)blocks), dim3(W * 64), 0, s, ev.start,
                              ev.stop, 0, g, t, q, out, base, n_q, st);
    return hipGetLastError();
}

}  // namespace pf

bool prefill_supported(const Geom &g) {
    return (g.d == 64 || g.d == 128) && g.kb >= 2 && g.kb <= 4 && g.vb >= 1 && g.vb <= 3 && g.norm_frac == 9 &&
           g.kv_shift == 0 && g.gq == 0;
}

hipError_t launch_attend_prefill(hipStream_t s, const Geom &g, const Tables *t, const int32_t *q, int32_t *out,
                                 int64_t base, int64_t n_q, int two_pass, LaunchEv ev, DevStats *st) {
    if (n_q <= 0) return hipSuccess;
    if (base < 0 || base + n_q > PREFILL_MAX_ROWS) return hipErrorInvalidValue;
    if (g.d == 64) {
        // A grid that fills the chip runs three workgroups a CU (32-token stages: 42 KB of LDS, 168
        // VGPRs); a smaller one has a CU each, and longer stages amortise their barriers.
        const bool few = n_q * g.G * g.n_kv < 32768;
        if (g.vb <= 2)
            return few ? pf::launch<64, 4, 4, 64>(s, g, t, q, out, base, n_q, two_pass, ev, st)
                       : pf::launch<64, 4, 4, 32>(s, g, t, q, out, base, n_q, two_pass, ev, st);
        return pf::launch<64, 8, 4, 32>(s, g, t, q, out, base, n_q, two_pass, ev, st);
    }
    if (g.vb <= 2) return pf::launch<128, 4, 8, 32>(s, g, t, q, out, base, n_q, two_pass, ev, st);
    return pf::launch<128, 8, 8, 32>(s, g, t, q, out, base, n_q, two_pass, ev, st);
}

}  // namespace insitu
