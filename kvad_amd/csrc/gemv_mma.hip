// Few-row matmul on the matrix cores: y[t][r] (+)= sum_b ws[r,b] xs[t,b]
// D_b[r,t] for a few to a few dozen token rows (Weight::matmul_bt,
// crates/llm/src/quant.rs:751-907, as forward_each calls it,
// llama.rs:418-434), q8 / q4 / Q4_K weights against the rows' int8 codes.
//
// D_b, the exact i32 dot of weight row r's 32-block b with token t's codes,
// is one v_mfma_i32_16x16x32_i8 for 16 weight rows x 16 tokens.  The block's
// scale products ws[r] xs[t] are an outer product, four blocks per
// v_mfma_f32_16x16x1_4b_f32 (block k from lanes 16k..16k+15 of both
// operands, its products in elements 4k..4k+3), so two VALU operations per
// output and block remain: convert the dot, fused multiply-add.  Q4_K's
// minimum terms sum_j dmin m_j[r] xs[t,j] sum_j[t] are a true product over
// the sub-block index: v_mfma_f32_16x16x4_f32, four sub-blocks an
// instruction, straight into the accumulators.
//
// What bounds it: the weights' stream, and at its ends the latency of the
// first loads.  A wave owns a fixed slice of the k-range, holds its slice of
// the codes and block scales of all 16 T tokens in registers in the matrix
// core's operand layout (the codes are read once per workgroup, not once per
// 16 weight rows), and walks the 16-row groups of its workgroup with D units
// of weights in flight in registers (a unit: 128 k-values of q8 / q4, a
// 256-wide Q4_K super-block).  KW waves share a group's k-range.
//
// Weights and codes come in with consecutive lanes on consecutive 16-byte
// pieces of a row and turn into the operand layout (a row per lane & 15)
// through a wave-private LDS stage.  Loads in the operand layout itself put
// every lane on a line of its own, which took the address units 43 cycles an
// instruction (s_memtime stamps), against 16.
//
// The waves' partial tiles meet in LDS in wave order (results do not depend on
// timing), double buffered, one barrier that waits on LDS only per group; the
// adds and the store fall to another wave each group.  Every load is
// unconditional (a lane with nothing to read addresses past its buffer's end,
// which reads zeros), so each wait covers only the loads it needs; bias and
// residual values are loaded ahead by the wave that will store the group.
//
// Measured (us per matmul under graph replay, the rows' quantisation launch of
// about 3 us included; against a kernel that loaded in the operand layout up
// to 8 tokens and the int8 GEMM above): Q4_K 14336x4096 at 5 / 12 / 32 / 64
// tokens 19.7 / 24.2 / 26.9 / 43.5 -> 13.8 / 14.0 / 19.5 / 30.8, 4096x14336
// 18.6 / 24.5 / 25.9 / 38.0 -> 15.7 / 16.2 / 22.4 / 37.3, 4096x4096 9.2 / 13.7
// / 16.2 / 19.5 -> 7.7 / 7.9 / 10.4 / 17.3; q8 4864x896 at 5 / 16 / 64 6.4 /
// 8.7 / 13.5 -> 5.8 / 5.9 / 8.7; q4 4096x4096 at 8 / 16 9.4 / 13.6 -> 7.7 /
// 7.8.  Eight waves of up to 256 registers a workgroup and one workgroup a CU
// beat sixteen of 128 (Q4_K 4096x4096 at 12 tokens 8.2 / 12.0, the registers
// spilling) and two workgroups a CU where a slice is more than a unit
// (14336x4096 13.9 / 16.8).
//
// Sums run in another order than the single-token GEMV's, so a token's row
// agrees with its matvec to rounding (1e-5 relative), not to the bit.
#include <algorithm>

#include "gemv_core.hpp"

namespace kh {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef unsigned long long u64;

constexpr unsigned OOB = 0xfff00000u;  // past every buffer here, immediate offsets included
constexpr int GROUP = 16;              // weight rows of a group, tokens of a tile

struct MmaJob {
    const void *w;
    const float *ws;     // q8 / q4 block scales [rows][nb]; unused for Q4_K
    const float *bias;   // [rows] or null
    float *y;            // [m][rows]
    int rows, accumulate;
    int wg0, nwg;        // the job's workgroups
};

struct MmaArgs {
    MmaJob j[MULTI_JOBS];
    // split z of the units (grid z, `per` units each) stores its sums to
    // part[z][all][rows] for a reduce launch, one job only; null: no split
    float *part;
    int per, all;
};

// What a launch runs on.
struct MmaRows {
    QAct x;  // the rows' codes, block scales and code sums (Q4_K's minimum term)
    int cols, m, njobs;
    int units;  // per row
};

// Keeps the compiler from moving this wave's LDS accesses across (LDS serves
// a wave's requests in order).
__device__ __forceinline__ void wave_order() { __asm__ volatile("" ::: "memory"); }

__device__ __forceinline__ u64 bld8(const rsrc_t &r, unsigned off) {
    return __builtin_bit_cast(u64, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
}

// A buffer descriptor over fewer than 2^32 bytes.
__device__ __forceinline__ rsrc_t rsrc32(const void *p, unsigned bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short)0, (int)bytes, RSRC_WORD3);
}

// Four nibble codes per byte lane -> signed (code - 8) bytes, no borrows.
__device__ __forceinline__ unsigned nib_minus8(unsigned x) {
    return ((x | 0x80808080u) - 0x08080808u) ^ 0x80808080u;
}
__device__ __forceinline__ u64 pack64(unsigned lo, unsigned hi) { return (u64)lo | ((u64)hi << 32); }

__device__ __forceinline__ v4i mma32(u64 a, u64 b) {
    const v4i z = {0, 0, 0, 0};
    return __builtin_amdgcn_mfma_i32_16x16x32_i8((long)a, (long)b, z, 0, 0, 0);
}

template <int PREC>
struct Shape {
    static constexpr int UK = PREC == KH_Q4K ? QK_K : 4 * BLOCK;  // k-values of a unit
    static constexpr int NB = UK / BLOCK, NQ = NB / 4;            // blocks, quads of blocks
};

// A stage row is a unit's codes of a weight row and 16 bytes of its scales:
// Q4_K's block as it lies (header, then codes), q8 / q4 codes, then four block
// scales.  Rows 36 (q4 20) banks apart serve the operand reads without
// conflicts.
template <int PREC>
struct RowStage {
    static constexpr int CB = PREC == KH_Q4 ? 64 : 128;  // bytes of codes
    static constexpr int STR = CB + 16;
    static constexpr int CODES = PREC == KH_Q4K ? 16 : 0, SCALES = PREC == KH_Q4K ? 0 : CB;
    static constexpr int RUN = PREC == KH_Q4K ? 9 : CB / 16;               // 16-byte pieces of a row in one run
    static constexpr int NL = (GROUP * RUN + WAVE - 1) / WAVE;             // loads a wave
};

// One unit of 16 weight rows in flight: piece i * 64 + lane of their runs,
// and for q8 / q4 row lane's four block scales (lanes 0-15).
template <int PREC>
struct Wts {
    int4 a[RowStage<PREC>::NL];
    int4 ws;
};

// A wave's slice of the tokens' codes and block scales, S units of T tiles of
// 16 tokens (token lane & 15, k-slot lane >> 4; scales of block lane >> 4).
template <int PREC, int S, int T>
struct Acts {
    u64 b[S][T][Shape<PREC>::NB];
    float xs[S][T][Shape<PREC>::NQ];
    float xm[PREC == KH_Q4K ? S : 1][T][Shape<PREC>::NQ];  // xs * code sum
};

// The first job's pointers and sizes lead the arguments (preloaded into
// scalar registers); gm: its workgroups << 16 | tokens.
template <int PREC, int KW, int S, int T, int D, int WPE, bool WIDE, bool SPLIT>
__global__ __launch_bounds__(WAVE *KW, WPE) void rows_mma_kernel(unsigned g12, unsigned gm, const void *w0,
                                                                 const float *ws0, const int8_t *xq, const float *xs,
                                                                 int rows0, int cols, const int32_t *xsum, MmaArgs a) {
    static_assert(MULTI_JOBS == 3, "g12 holds jobs 1 and 2");
    constexpr int UK = Shape<PREC>::UK, NB = Shape<PREC>::NB, NQ = Shape<PREC>::NQ;
    using RS = RowStage<PREC>;
    constexpr int XSTR = UK + 16;  // a token's stage row
    constexpr int STAGE = GROUP * (XSTR > 16 * S * NQ ? XSTR : 16 * S * NQ);
    static_assert(XSTR >= RS::STR, "the stage holds a unit of weights too");
    __shared__ __align__(16) v4f s_red[2][KW][T][WAVE];
    __shared__ __align__(16) char s_stage[KW][STAGE];
    const int tid = threadIdx.x, lane = tid & (WAVE - 1), lr = lane & 15, lg = lane >> 4;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ji = ((int)blockIdx.x >= (int)(g12 & 0xffffu) ? 1 : 0) + ((int)blockIdx.x >= (int)(g12 >> 16) ? 1 : 0);
    const MmaJob &job = a.j[ji];
    const void *wp = w0;
    const float *wsp = ws0;
    int rows = rows0;
    unsigned wg = blockIdx.x, step = gm >> 16;
    if (ji) {
        wp = job.w, wsp = job.ws, rows = job.rows;
        wg -= (unsigned)job.wg0, step = (unsigned)job.nwg;
    }
    const unsigned nb = (unsigned)cols / BLOCK, groups = ((unsigned)rows + GROUP - 1) / GROUP;
    unsigned units = ((unsigned)cols + UK - 1) / UK, first = 0;
    if constexpr (SPLIT) {
        first = blockIdx.z * (unsigned)a.per;
        units = min(units - first, (unsigned)a.per);
    }
    const int t0 = (int)blockIdx.y * GROUP * T, m = (int)(gm & 0xffffu) - t0;
    const unsigned mt = (unsigned)min(m, GROUP * T);  // this workgroup's tokens
    const unsigned row_bytes = PREC == KH_Q8 ? (unsigned)cols
                               : PREC == KH_Q4 ? (unsigned)cols / 2
                                               : (unsigned)cols / QK_K * Q4K_BYTES;
    constexpr unsigned UB = PREC == KH_Q4K ? Q4K_BYTES : RS::CB;  // a unit's bytes of a row
    // (sizes fit 32 bits: mma_addresses)
    const rsrc_t X = rsrc32(xq + (size_t)t0 * cols, mt * (unsigned)cols);
    const rsrc_t XS = rsrc32(xs + (size_t)t0 * nb, mt * nb * 4);
    const rsrc_t XM = rsrc32(xsum + (size_t)t0 * nb, mt * nb * 4);
    const rsrc_t W = rsrc32(wp, (unsigned)rows * row_bytes);
    const rsrc_t WS = rsrc32(wsp, PREC == KH_Q4K ? 0 : (unsigned)rows * nb * 4);
    char *const st = s_stage[wv];

    // k-ranges of KW * S units in turn (WIDE), or one
    for (unsigned c0 = 0; c0 < (WIDE ? units : 1u); c0 += KW * S) {
        const unsigned U = WIDE ? min(units - c0, (unsigned)(KW * S)) : units;
        const unsigned u0 = first + c0 + U * wv / KW, cnt = first + c0 + U * (wv + 1) / KW - u0;  // this wave's units

        // The tokens' codes in 16-byte pieces, then their scales and code
        // sums, 16 bytes (four blocks) a piece.  Units past the wave's share
        // are never used and tokens past m lie past the buffers' ends.
        constexpr int XL = UK / 64;                              // code loads of a unit of 16 tokens
        constexpr int SP = S * NQ, SL = (GROUP * SP + WAVE - 1) / WAVE;  // scale pieces a token, loads
        int4 rx[S][T][XL], rs[SL][T], rm[PREC == KH_Q4K ? SL : 1][T];
#pragma unroll
        for (int u = 0; u < S; u++)
#pragma unroll
            for (int tt = 0; tt < T; tt++)
#pragma unroll
                for (int i = 0; i < XL; i++) {
                    const unsigned p = i * WAVE + lane, tok = tt * GROUP + p / (UK / 16), k = (u0 + u) * UK + 16 * (p % (UK / 16));
                    const unsigned o = tok * (unsigned)cols + k;
                    rx[u][tt][i] = bld16(X, PREC == KH_Q4K || k < (unsigned)cols ? o : OOB);  // a k tail is zero codes
                }
#pragma unroll
        for (int tt = 0; tt < T; tt++)
#pragma unroll
            for (int i = 0; i < SL; i++) {
                const unsigned p = i * WAVE + lane, tok = tt * GROUP + p / SP;
                const unsigned o = SL * WAVE == GROUP * SP || p < GROUP * SP ? (tok * nb + u0 * NB + 4 * (p % SP)) * 4 : OOB;
                rs[i][tt] = bld16(XS, o);
                if constexpr (PREC == KH_Q4K) rm[i][tt] = bld16(XM, o);
            }
        __builtin_amdgcn_sched_barrier(0);

        // this lane's pieces of a group's rows, from the group's first row
        unsigned lw[RS::NL];
#pragma unroll
        for (int i = 0; i < RS::NL; i++) {
            const unsigned p = i * WAVE + lane;
            lw[i] = p / RS::RUN * row_bytes + u0 * UB + 16 * (p % RS::RUN);
            if (RS::NL * WAVE != GROUP * RS::RUN && p >= GROUP * RS::RUN) lw[i] = OOB;
        }
        const unsigned lws = lane < GROUP ? ((unsigned)lane * nb + u0 * NB) * 4 : OOB;
        auto load = [&](Wts<PREC> &w, unsigned group, int u) {
            // a unit past the wave's share, or a lane without a piece, reads
            // past the end; a group past the last does by itself
            const unsigned base = (unsigned)u < cnt ? group * GROUP * row_bytes + u * UB : OOB;
#pragma unroll
            for (int i = 0; i < RS::NL; i++) w.a[i] = bld16(W, max(base, lw[i]) >= OOB ? OOB : base + lw[i]);
            if constexpr (PREC != KH_Q4K) {
                const unsigned bs = (unsigned)u < cnt ? group * GROUP * nb * 4 + u * NB * 4 : OOB;
                w.ws = bld16(WS, max(bs, lws) >= OOB ? OOB : bs + lws);
            }
        };
        Wts<PREC> w[D];
#pragma unroll
        for (int i = 0; i < D; i++) load(w[i], wg + (i / S) * step, i % S);
        __builtin_amdgcn_sched_barrier(0);

        // the scales, then the codes, through the wave's stage into the
        // operand layout
        Acts<PREC, S, T> x;
#pragma unroll
        for (int tt = 0; tt < T; tt++)
#pragma unroll
            for (int u = 0; u < S; u++) {
#pragma unroll
                for (int i = 0; i < XL; i++) {
                    const int p = i * WAVE + lane;
                    *reinterpret_cast<int4 *>(st + (p / (UK / 16)) * XSTR + 16 * (p % (UK / 16))) = rx[u][tt][i];
                }
                wave_order();
#pragma unroll
                for (int k = 0; k < NB; k++) {
                    if constexpr (PREC == KH_Q4) {
                        // byte i of a weight block: weight i (low nibble), 16 + i (high)
                        const char *p = st + lr * XSTR + 32 * k + 4 * lg;
                        x.b[u][tt][k] = pack64(*reinterpret_cast<const unsigned *>(p),
                                               *reinterpret_cast<const unsigned *>(p + 16));
                    } else {
                        x.b[u][tt][k] = *reinterpret_cast<const u64 *>(st + lr * XSTR + 32 * k + 8 * lg);
                    }
                }
                wave_order();
            }
#pragma unroll
        for (int tt = 0; tt < T; tt++)
#pragma unroll
            for (int pass = 0; pass < (PREC == KH_Q4K ? 2 : 1); pass++) {
#pragma unroll
                for (int i = 0; i < SL; i++)
                    if (SL * WAVE == GROUP * SP || i * WAVE + lane < GROUP * SP)
                        *reinterpret_cast<int4 *>(st + (i * WAVE + lane) * 16) = pass ? rm[i][tt] : rs[i][tt];
                wave_order();
#pragma unroll
                for (int u = 0; u < S; u++)
#pragma unroll
                    for (int q = 0; q < NQ; q++) {
                        const char *p = st + (lr * SP + u * NQ + q) * 16 + 4 * lg;
                        if (pass == 0) {
                            const float v = *reinterpret_cast<const float *>(p);
                            x.xs[u][tt][q] = PREC == KH_Q4K || (u0 + u) * NB + 4 * q + lg < nb ? v : 0.0f;
                        } else if constexpr (PREC == KH_Q4K) {
                            x.xm[u][tt][q] = x.xs[u][tt][q] * (float)*reinterpret_cast<const int *>(p);
                        }
                    }
                wave_order();
            }

        v4f acc[T];
#pragma unroll
        for (int tt = 0; tt < T; tt++) acc[tt] = v4f{0.f, 0.f, 0.f, 0.f};
        auto stage = [&](const Wts<PREC> &w) {
#pragma unroll
            for (int i = 0; i < RS::NL; i++) {
                const int p = i * WAVE + lane;
                if (RS::NL * WAVE == GROUP * RS::RUN || p < GROUP * RS::RUN)
                    *reinterpret_cast<int4 *>(st + (p / RS::RUN) * RS::STR + 16 * (p % RS::RUN)) = w.a[i];
            }
            if constexpr (PREC != KH_Q4K)
                if (lane < GROUP) *reinterpret_cast<int4 *>(st + lane * RS::STR + RS::SCALES) = w.ws;
            wave_order();
        };
        auto compute = [&](int u) {
            const char *const sr = st + lr * RS::STR;
            int4 h;
            float d, dmin;
            if constexpr (PREC == KH_Q4K) {
                h = *reinterpret_cast<const int4 *>(sr);
                d = half_bits_to_float((unsigned)h.x), dmin = half_bits_to_float((unsigned)h.x >> 16);
            }
            // the unit's own sum, added to the group's once: shorter chains (the
            // error against 64 bits at 12 rows, 2-norm, one chain / these: Q4_K
            // 4096x14336 2.25e-7 / 1.50e-7, 14336x4096 1.54e-7 / 1.39e-7, q8
            // 4096x14336 1.49e-7 / 1.03e-7; Q4_K 4096x14336 15.6 -> 16.2 us, every
            // other time the same)
            v4f sum[T];
#pragma unroll
            for (int tt = 0; tt < T; tt++) sum[tt] = v4f{0.f, 0.f, 0.f, 0.f};
            // four blocks at a time: their operands, scale products and dots
            // are the only ones live
#pragma unroll
            for (int q = 0; q < NQ; q++) {
                float sc, mn;
                u64 A[4];
                if constexpr (PREC == KH_Q4K) {
                    // sub-block lg + 4q of row lr: d * sc and dmin * m (mpp.rs:276-282, 304-315)
                    unsigned s6, m6;
                    q4k_scale_min_bfe(h, q4k_lane(lg + 4 * q), s6, m6);
                    sc = d * (float)s6;
                    mn = -(dmin * (float)m6);
#pragma unroll
                    for (int c = 0; c < 2; c++) {
                        const u64 v = *reinterpret_cast<const u64 *>(sr + RS::CODES + 64 * q + 32 * c + 8 * lg);
                        const unsigned lo = (unsigned)v, hi = (unsigned)(v >> 32);
                        A[2 * c] = pack64(lo & 0x0f0f0f0fu, hi & 0x0f0f0f0fu);
                        A[2 * c + 1] = pack64((lo >> 4) & 0x0f0f0f0fu, (hi >> 4) & 0x0f0f0f0fu);
                    }
                } else {
                    // past the row's last block the stage holds the next row's
                    // scale: kept out (its codes meet zero codes)
                    const float v = *reinterpret_cast<const float *>(sr + RS::SCALES + 4 * lg);
                    sc = (u0 + u) * NB + lg < nb ? v : 0.0f;
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        if constexpr (PREC == KH_Q8) {
                            A[k] = *reinterpret_cast<const u64 *>(sr + 32 * k + 8 * lg);
                        } else {
                            const unsigned c = *reinterpret_cast<const unsigned *>(sr + 16 * k + 4 * lg);
                            A[k] = pack64(nib_minus8(c & 0x0f0f0f0fu), nib_minus8((c >> 4) & 0x0f0f0f0fu));
                        }
                    }
                }
#pragma unroll
                for (int tt = 0; tt < T; tt++) {
                    const v16f z16 = {};
                    const v16f P = __builtin_amdgcn_mfma_f32_16x16x1f32(sc, x.xs[u][tt][q], z16, 0, 0, 0);
                    v4i Dv[4];
#pragma unroll
                    for (int k = 0; k < 4; k++) Dv[k] = mma32(A[k], x.b[u][tt][4 * q + k]);
                    if constexpr (PREC == KH_Q4K)
                        sum[tt] = __builtin_amdgcn_mfma_f32_16x16x4f32(mn, x.xm[u][tt][q], sum[tt], 0, 0, 0);
#pragma unroll
                    for (int k = 0; k < 4; k++)
#pragma unroll
                        for (int i = 0; i < 4; i++) sum[tt][i] = fmaf(P[4 * k + i], (float)Dv[k][i], sum[tt][i]);
                    if constexpr (NQ * T > 1) __builtin_amdgcn_sched_barrier(0);
                }
            }
#pragma unroll
            for (int tt = 0; tt < T; tt++) acc[tt] += sum[tt];
        };

        const bool plain = !SPLIT || !a.part;
        float *yp = job.y + (size_t)t0 * rows;
        if (!plain) yp = a.part + ((size_t)blockIdx.z * a.all + t0) * rows;
        const bool add_old = (plain && job.accumulate) || (WIDE && c0 > 0), add_bias = plain && job.bias && !(WIDE && c0 > 0);
        const rsrc_t BI = rsrc32(job.bias, add_bias && !add_old ? (unsigned)rows * 4 : 0);
        const rsrc_t Y = rsrc32(yp, mt * (unsigned)rows * 4);
        // steps run through the groups' units; buffer i takes steps i, i + D,
        // ...: an unrolled body of TB groups brings the buffers round
        constexpr int TB = D % S == 0 ? D / S : S % D == 0 ? 1 : D;
        static_assert((TB * S) % D == 0, "whole rounds of buffers a body");
        int it = 0;  // groups done: which wave adds and stores, which buffer
        for (unsigned g = wg; g < groups; g += TB * step) {
#pragma unroll
            for (int tb = 0; tb < TB; tb++) {
                const unsigned group = g + tb * step;
                if (group >= groups) break;
                v4f ex[T];  // what the group's stores add: the old values, else the bias
#pragma unroll
                for (int tt = 0; tt < T; tt++) {
                    const bool mine = (it * T + tt) % KW == wv;
                    const unsigned ro = (group * GROUP + 4 * lg) * 4;
                    const unsigned tok = (unsigned)(tt * GROUP + lr);
                    const unsigned o = add_old ? tok * (unsigned)rows * 4 + ro : ro;
                    ex[tt] = __builtin_bit_cast(v4f, bld16f(add_old ? Y : BI, mine ? o : OOB));
                }
#pragma unroll
                for (int u = 0; u < S; u++) {
                    const int i = tb * S + u;
                    if ((unsigned)u < cnt) stage(w[i % D]);
                    load(w[i % D], group + ((u + D) / S) * step, (u + D) % S);
                    if ((unsigned)u < cnt) compute(u);
                    wave_order();
                }
                // the group's partial tiles: summed and stored by one wave a tile
#pragma unroll
                for (int tt = 0; tt < T; tt++) {
                    s_red[it & 1][wv][tt][lane] = acc[tt];
                    acc[tt] = v4f{0.f, 0.f, 0.f, 0.f};
                }
                __asm__ volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
                for (int tt = 0; tt < T; tt++) {
                    if ((it * T + tt) % KW != wv) continue;
                    v4f s = s_red[it & 1][0][tt][lane];
#pragma unroll
                    for (int k = 1; k < KW; k++) s += s_red[it & 1][k][tt][lane];
                    if (add_bias && add_old) {  // (no caller passes both: loaded here)
#pragma unroll
                        for (int i = 0; i < 4; i++)
                            if ((int)group * GROUP + 4 * lg + i < rows) s[i] += job.bias[group * GROUP + 4 * lg + i];
                    }
                    // finish, quant.rs:849-858; x += proj (llama.rs:273-276)
                    if (add_bias || add_old) s = ex[tt] + s;
                    const int tok = tt * GROUP + lr, r = (int)group * GROUP + 4 * lg;
                    const unsigned off = ((unsigned)tok * (unsigned)rows + (unsigned)r) * 4;
                    if (tok < m) {
                        if (r + 3 < rows) {
                            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4i, s), Y, off, 0, 0);
                        } else {
#pragma unroll
                            for (int i = 0; i < 3; i++) {
                                const float v = s[i];  // (a bit cast of the element itself takes element 0)
                                if (r + i < rows)
                                    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(int, v), Y, off + 4 * i, 0,
                                                                          0);
                            }
                        }
                    }
                }
                it++;
            }
        }
        if constexpr (WIDE) __syncthreads();  // the next k-range adds into what this one stored
    }
}

// (waves along k, units a wave, tiles of 16 tokens, units in flight, waves a SIMD)
template <int PREC, int KW, int S, int T, int D, int WPE, bool WIDE = false, bool SPLIT = false>
int launch_rows(kh_ctx *ctx, const MmaRows &r, MmaArgs a, unsigned gz = 1) {
    const int cu = ctx->cu_count > 0 ? ctx->cu_count : 256;
    // as many workgroups as the CUs hold at WPE waves a SIMD, each job its
    // share by rows, at least one
    long long total = 0;
    for (int i = 0; i < r.njobs; i++) total += (a.j[i].rows + GROUP - 1) / GROUP;
    // one workgroup per CU, two where a one-unit slice leaves the registers
    // for it and there are groups enough to keep both busy (q8 151936x896 at
    // 8 rows 36.0 -> 34.1 us; 4864x896, 304 groups, 5.8 -> 6.1)
    const int slots = cu * (4 * WPE / KW) * (S == 1 && total >= 8LL * cu ? 2 : 1) / (int)gz;
    int nwg = 0;
    for (int i = 0; i < r.njobs; i++) {
        const int groups = (a.j[i].rows + GROUP - 1) / GROUP;
        int n = total <= slots ? groups : (int)((long long)slots * groups / total);
        n = n < 1 ? 1 : n > groups ? groups : n;
        a.j[i].wg0 = nwg;
        a.j[i].nwg = n;
        nwg += n;
    }
    if (nwg >= 0xffff) return fail(KH_DECLINED, "matmul: 65535 workgroups or more in one launch");
    const unsigned gy = (unsigned)((r.m + GROUP * T - 1) / (GROUP * T));
    const unsigned gm = (unsigned)a.j[0].nwg << 16 | (unsigned)r.m;
    hipLaunchKernelGGL((rows_mma_kernel<PREC, KW, S, T, D, WPE, WIDE, SPLIT>), dim3((unsigned)nwg, gy, gz), dim3(WAVE * KW), 0,
                       ctx->stream, multi_firsts(r.njobs, a.j[1].wg0, a.j[2].wg0), gm, a.j[0].w, a.j[0].ws, r.x.qs,
                       r.x.scales, a.j[0].rows, r.cols, r.x.sums, a);
    KH_HIP(hipGetLastError());
    return KH_OK;
}

// Units split over grid z, 8 * S a split: wide rows at more than 16 tokens,
// whose codes a wave's registers cannot hold for the whole width.
template <int PREC, int S>
int launch_split(kh_ctx *ctx, const MmaRows &r, MmaArgs a) {
    const unsigned gz = (unsigned)((r.units + 8 * S - 1) / (8 * S));
    a.per = (int)((r.units + gz - 1) / gz);
    a.all = r.m;
    const MmaJob j = a.j[0];
    int rc = launch_rows<PREC, 8, S, 2, 4, 2, false, true>(ctx, r, a, gz);
    if (rc) return rc;
    return launch_split_reduce(ctx, a.part, (int)gz, r.m, j.rows, j.bias, j.accumulate, j.y);
}

template <int PREC, int T>
int launch_units(kh_ctx *ctx, const MmaRows &r, MmaArgs a) {
    const int U = r.units;
    if constexpr (T == 2) {
        constexpr int S = PREC == KH_Q4K ? 2 : 4;
        if (U > 8 * S && r.njobs == 1) {
            const size_t gz = (size_t)(U + 8 * S - 1) / (8 * S);
            a.part = split_partials(ctx, gz * r.m * a.j[0].rows * 4);
            if (a.part) return launch_split<PREC, S>(ctx, r, a);
        }
    }
    if (U <= 4) return launch_rows<PREC, 4, 1, T, 3, 2>(ctx, r, a);
    if (U <= 8) return launch_rows<PREC, 8, 1, T, 3, 2>(ctx, r, a);
    if (U <= 16) return launch_rows<PREC, 8, 2, T, 4, 2>(ctx, r, a);
    if constexpr (PREC == KH_Q4K) {
        if (U <= 32) return launch_rows<PREC, 8, 4, 1, 4, 2>(ctx, r, a);
        return launch_rows<PREC, 8, 7, 1, 2, 2, true>(ctx, r, a);
    } else {
        if (U <= 32) return launch_rows<PREC, 8, 4, T, 4, 2>(ctx, r, a);
        if (U <= 64) return launch_rows<PREC, 8, 8, 1, 4, 2>(ctx, r, a);
        return launch_rows<PREC, 8, 14, 1, 2, 2, true>(ctx, r, a);
    }
}

template <int PREC>
int launch_prec(kh_ctx *ctx, const MmaRows &r, const MmaArgs &a) {
    return r.m <= GROUP ? launch_units<PREC, 1>(ctx, r, a) : launch_units<PREC, 2>(ctx, r, a);
}

}  // namespace

int launch_gemv_mma(kh_ctx *ctx, int njobs, const kh_weight *const *w, const float *const *bias, float *const *y,
                    const int *accumulate, const QAct &x, size_t m) {
    if (m == 0) return KH_OK;
    if (njobs < 1 || njobs > MULTI_JOBS) return fail(KH_EINVAL, "matmul: one to three weights per launch");
    const int prec = w[0]->precision;
    const size_t cols = w[0]->cols;
    if (prec != KH_Q8 && prec != KH_Q4 && prec != KH_Q4K)
        return fail(KH_EINVAL, "matmul: the matrix-core GEMV takes quantised weights");
    if (cols % (prec == KH_Q4K ? QK_K : BLOCK)) return fail(KH_EINVAL, "matmul: width not a whole number of blocks");
    MmaArgs a{};
    const int nb = (int)(cols / BLOCK);
    MmaRows r{QAct{}, (int)cols, 0, njobs, prec == KH_Q4K ? (int)(cols / QK_K) : (nb + 3) / 4};
    for (int i = 0; i < njobs; i++) {
        if (w[i]->precision != prec || w[i]->cols != cols)
            return fail(KH_EINVAL, "matmul: weights of one launch share precision and width");
        if (!mma_addresses(prec, w[i]->rows, cols))
            return fail(KH_DECLINED, "matmul: operands of 4 GiB or more are not addressed here");
        a.j[i] = MmaJob{w[i]->qs, w[i]->scales, bias ? bias[i] : nullptr, y[i], (int)w[i]->rows,
                        accumulate ? accumulate[i] : 0, 0, 0};
    }
    // tokens a launch: a 16-bit count
    const size_t step = 32768;
    for (size_t t0 = 0; t0 < m; t0 += step) {
        MmaArgs b = a;
        r.m = (int)std::min(m - t0, step);
        r.x = QAct{x.qs + t0 * cols, x.scales + t0 * nb, x.sums + t0 * nb};
        for (int i = 0; i < njobs; i++) b.j[i].y = a.j[i].y + t0 * a.j[i].rows;
        int rc;
        switch (prec) {
            case KH_Q8: rc = launch_prec<KH_Q8>(ctx, r, b); break;
            case KH_Q4: rc = launch_prec<KH_Q4>(ctx, r, b); break;
            default: rc = launch_prec<KH_Q4K>(ctx, r, b); break;
        }
        if (rc) return rc;
    }
    return KH_OK;
}

bool mma_addresses(int prec, size_t rows, size_t cols) {
    const size_t rb = prec == KH_Q8 ? cols : prec == KH_Q4 ? cols / 2 : cols / QK_K * Q4K_BYTES;
    // the last group's overhang (up to 15 rows) included; 32 tokens' outputs
    return (rows + 16) * rb < OOB && (rows + 16) * (cols / BLOCK) * 4 < OOB && 32 * rows * 4 < OOB && 32 * cols < ((size_t)1 << 31);
}

}  // namespace kh
