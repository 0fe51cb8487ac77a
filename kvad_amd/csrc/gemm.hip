// Batched prefill GEMM on CDNA4 matrix cores: Weight::matmul_bt
// (crates/llm/src/quant.rs:751-907, x86 row_dot path) for q8 / q4 / Q4_K
// weights, and tensor::gemm_bt (tensor.rs:102-186) for f32 weights.
//
// Quantised weights.  y[m, r] = sum_b ws[r,b] * xs[m,b] * D_b[r,m] where
// D_b is the exact i32 dot of weight row r's 32-block b with token m's
// quantised block (row_dot pass 1, quant.rs:876-897).  One
// v_mfma_i32_32x32x32_i8 computes D_b for a 32x32 (rows x tokens) tile and
// exactly one 32-wide block, so every block dot is the reference's integer;
// the block's scaling (pass 2, quant.rs:899-905) is applied to the tile in
// registers before the next block.  q4 nibbles are widened to (code - 8) in
// LDS (the same integers as q4_row_dots, quant.rs:168-189); Q4_K codes are
// widened unsigned and their sub-block scale/min terms applied as the GEMV
// does (y += xs * (d*sc*dot - dmin*m*sum), mpp.rs:304-315).
//
// The per-block scaling is the bound: with 32-wide scale blocks on both
// operands every output takes a scaled term per block.  The scale products
// ws[r] * xs[t] of a tile are an outer product, computed on the matrix core,
// two tiles per v_mfma_f32_32x32x1_2b_f32 (half the matrix-core time of one
// 32x32x2 product per tile with a k-slot zeroed); Q4_K's minimum terms
// sum_b dmin*m * xs*sum are a true product over the block index and go into
// the accumulators by MFMA as well.  Two VALU operations per output per
// block remain (convert the i32 dot, fused multiply-add); matrix-core
// results are kept in VGPRs (-mllvm -amdgpu-mfma-vgpr-form), where the
// epilogue reads them without a copy.
//
// Tiles.  A workgroup of 4 waves computes a BN x BM (weight rows x tokens)
// tile; each wave WR/WT-splits it into RT x TT MFMA tiles of 32 x 32.  A
// stage is 128 k-values (4 blocks): weight and activation bytes go global ->
// registers (next stage, in flight during compute) -> LDS (rows padded by 16
// bytes), with the stage's scales beside them.  Buffer loads return zeros
// past the end of an array, so edge tiles need no branches on rows or
// tokens; a k tail (K % 128 != 0) is masked explicitly.
//
// f32 weights use v_mfma_f32_32x32x2_f32 over 32-wide k stages with the same
// tile map.  Sums are taken in a different order from the reference's
// 4-lane register tiles, so results agree to rounding (1e-5 relative).
#include <algorithm>

#include "common.hpp"

namespace kh {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v32f __attribute__((ext_vector_type(32)));


constexpr unsigned RSRC_WORD3 = 0x00020000;  // raw buffer, gfx9 family
typedef __amdgpu_buffer_rsrc_t rsrc_t;

__device__ __forceinline__ rsrc_t rsrc(const void *p, size_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short)0,
                                             (int)(bytes > 0xffffffffu ? 0xffffffffu : bytes), RSRC_WORD3);
}
__device__ __forceinline__ int4 ld16(const rsrc_t &r, unsigned off) {
    return __builtin_bit_cast(int4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}
__device__ __forceinline__ float ldf(const rsrc_t &r, unsigned off) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
}
__device__ __forceinline__ int ldi(const rsrc_t &r, unsigned off) {
    return (int)__builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0);
}

__device__ __forceinline__ float half_bits_to_float(unsigned h) {
    return (float)__builtin_bit_cast(_Float16, (unsigned short)(h & 0xffff));
}

// Four nibble codes per byte lane -> signed (code - 8) bytes, no borrows.
__device__ __forceinline__ int nib_minus8(int x) {
    return (int)((((unsigned)x | 0x80808080u) - 0x08080808u) ^ 0x80808080u);
}


constexpr int THREADS = 256;
constexpr int BK = 128;              // k per stage (bytes of int8)
constexpr int NBS = BK / BLOCK;      // 32-blocks per stage
constexpr int ASTR = BK + 16;        // LDS row stride, bytes

// A wave's RT x TT tiles when all of them lie inside the output (and the
// output and bias are 16-byte aligned with rows a multiple of 4 wide): one
// float4 per four rows, no per-element bounds and no branches.  dst is the
// output (bias and accumulate as store_tiles) or a split's partial plane
// (neither).  Returns false, having written nothing, otherwise.
template <int RT, int TT>
__device__ __forceinline__ bool store_tiles_full(const GemmArgs &a, float *dst, bool partial, const v16f (&acc)[RT][TT],
                                                 int r_base, int t_base, int t_end, int lane) {
    const float *bias = partial ? nullptr : a.bias;
    const bool accumulate = !partial && a.accumulate;
    if ((a.N & 3) || r_base + RT * 32 > a.N || t_base + TT * 32 > t_end ||
        (((uintptr_t)dst | (uintptr_t)bias) & 15))
        return false;
    const rsrc_t Y = rsrc(dst + (size_t)t_base * a.N + r_base, ((size_t)(TT * 32 - 1) * a.N + RT * 32) * 4);
    float4 bv[RT][4];
#pragma unroll
    for (int rt = 0; rt < RT; rt++)
#pragma unroll
        for (int g = 0; g < 4; g++)
            bv[rt][g] = bias ? *reinterpret_cast<const float4 *>(bias + r_base + rt * 32 + 8 * g + 4 * (lane >> 5))
                             : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int rt = 0; rt < RT; rt++)
#pragma unroll
        for (int tt = 0; tt < TT; tt++)
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const unsigned off = ((unsigned)(tt * 32 + (lane & 31)) * (unsigned)a.N +
                                      (unsigned)(rt * 32 + 8 * g + 4 * (lane >> 5))) * 4u;
                float4 v = make_float4(acc[rt][tt][4 * g], acc[rt][tt][4 * g + 1], acc[rt][tt][4 * g + 2],
                                       acc[rt][tt][4 * g + 3]);
                if (!partial) {  // + bias (0 without one), finish, quant.rs:849-858
                    const float4 b = bv[rt][g];
                    v = make_float4(v.x + b.x, v.y + b.y, v.z + b.z, v.w + b.w);
                }
                if (accumulate) {  // x += proj (llama.rs:273-276)
                    const float4 o = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(Y, off, 0, 0));
                    v = make_float4(o.x + v.x, o.y + v.y, o.z + v.z, o.w + v.w);
                }
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4i, v), Y, off, 0, 0);
            }
    return true;
}

// Writes a 32x32 accumulator tile (lane: token l&31, rows 8g + 4(l>>5) + e).
template <int RT, int TT>
__device__ __forceinline__ void store_tiles(const GemmArgs &a, const v16f (&acc)[RT][TT], int r_base, int t_base,
                                            int t_end, int lane) {
    if (store_tiles_full<RT, TT>(a, a.y, false, acc, r_base, t_base, t_end, lane)) return;
    const bool vec = (a.N & 3) == 0;
#pragma unroll
    for (int rt = 0; rt < RT; rt++)
#pragma unroll
        for (int tt = 0; tt < TT; tt++) {
            const int tok = t_base + tt * 32 + (lane & 31);
            if (tok >= t_end) continue;
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const int r = r_base + rt * 32 + 8 * g + 4 * (lane >> 5);
                float v[4];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const float add = a.bias && r + e < a.N ? a.bias[r + e] : 0.0f;  // finish, quant.rs:849-858
                    v[e] = acc[rt][tt][4 * g + e] + add;
                }
                float *dst = a.y + (size_t)tok * a.N + r;
                if (vec && r + 3 < a.N) {
                    if (a.accumulate) {  // x += proj (llama.rs:273-276)
                        const float4 o = *reinterpret_cast<const float4 *>(dst);
                        v[0] = o.x + v[0], v[1] = o.y + v[1], v[2] = o.z + v[2], v[3] = o.w + v[3];
                    }
                    *reinterpret_cast<float4 *>(dst) = make_float4(v[0], v[1], v[2], v[3]);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        if (r + e < a.N) dst[e] = a.accumulate ? dst[e] + v[e] : v[e];
                }
            }
        }
}

// Split-K: split z writes its tile's sums, unscaled by bias or residual, to
// part[z][M][N]; split_reduce_kernel, launched next, adds the splits.
template <int RT, int TT>
__device__ __forceinline__ void store_partials(const GemmArgs &a, const v16f (&acc)[RT][TT], int r_base, int t_base,
                                               int t_end, int lane) {
    const size_t plane = (size_t)a.M * a.N;
    float *part = a.part + blockIdx.z * plane;
    if (store_tiles_full<RT, TT>(a, part, true, acc, r_base, t_base, t_end, lane)) return;
    const bool vec = (a.N & 3) == 0;
#pragma unroll
    for (int rt = 0; rt < RT; rt++)
#pragma unroll
        for (int tt = 0; tt < TT; tt++) {
            const int tok = t_base + tt * 32 + (lane & 31);
            if (tok >= t_end) continue;
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const int r = r_base + rt * 32 + 8 * g + 4 * (lane >> 5);
                float *dst = part + (size_t)tok * a.N + r;
                if (vec && r + 3 < a.N) {
                    *reinterpret_cast<float4 *>(dst) = make_float4(acc[rt][tt][4 * g], acc[rt][tt][4 * g + 1],
                                                                   acc[rt][tt][4 * g + 2], acc[rt][tt][4 * g + 3]);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        if (r + e < a.N) dst[e] = acc[rt][tt][4 * g + e];
                }
            }
        }
}

// Split-K's second launch: y = part[0] + part[1] + ... (split order), then
// bias and residual as store_tiles.  One thread per four outputs.
__global__ __launch_bounds__(256) void split_reduce_kernel(const float *part, int ks, int M, int N,
                                                           const float *bias, int accumulate, float *y) {
    const size_t plane = (size_t)M * N, e0 = ((size_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (e0 >= plane) return;
    if ((N & 3) == 0) {  // the four outputs share a token
        const rsrc_t PT = rsrc(part, (size_t)ks * plane * 4);
        const unsigned o = (unsigned)(e0 * 4), step = (unsigned)(plane * 4);
        // every split's load in flight at once (up to 32; those past ks read
        // outside the buffer, as zeros), then the adds in split order
        float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
        for (int z0 = 0; z0 < ks; z0 += 32) {
            float4 p[32];
#pragma unroll
            for (int j = 0; j < 32; j++)
                p[j] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(
                                                      PT, z0 + j < ks ? o + (z0 + j) * step : 0xffffffffu, 0, 0));
#pragma unroll
            for (int j = 0; j < 32; j++)
                if (z0 + j < ks) x = make_float4(x.x + p[j].x, x.y + p[j].y, x.z + p[j].z, x.w + p[j].w);
        }
        const int r = (int)(e0 % N);
        float v[4] = {x.x, x.y, x.z, x.w};
        if (bias) {  // finish, quant.rs:849-858
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] = v[e] + bias[r + e];
        }
        float4 *dst = reinterpret_cast<float4 *>(y + e0);
        if (accumulate) {  // x += proj (llama.rs:273-276)
            const float4 o4 = *dst;
            v[0] = o4.x + v[0], v[1] = o4.y + v[1], v[2] = o4.z + v[2], v[3] = o4.w + v[3];
        }
        *dst = make_float4(v[0], v[1], v[2], v[3]);
        return;
    }
    for (int e = 0; e < 4 && e0 + e < plane; e++) {
        float x = 0.f;
        for (int z = 0; z < ks; z++) x = x + part[z * plane + e0 + e];
        const int r = (int)((e0 + e) % N);
        if (bias) x = x + bias[r];
        y[e0 + e] = accumulate ? y[e0 + e] + x : x;
    }
}

// ---------------------------------------------------------------------------
// int8 MFMA GEMM for q8 / q4 / Q4_K weights
// ---------------------------------------------------------------------------

template <int PREC, int WR, int WT, int RT, int TT>
__global__ __launch_bounds__(THREADS) void gemm_i8_kernel(GemmArgs a) {
    static_assert(WR * WT == 4, "four waves");
    constexpr int BN = WR * RT * 32, BM = WT * TT * 32;
    // per-thread global chunk counts of one stage
    constexpr int A_CH = PREC == KH_Q8 ? BN * (BK / 16) : BN * NBS;  // q4 / Q4_K: one 16-byte chunk per block
    constexpr int A_PT = (A_CH + THREADS - 1) / THREADS;
    constexpr int B_CH = BM * (BK / 16);
    constexpr int B_PT = (B_CH + THREADS - 1) / THREADS;
    constexpr int WS_PT = (BN * NBS + THREADS - 1) / THREADS;
    constexpr int XS_PT = (BM * NBS + THREADS - 1) / THREADS;

    __shared__ __align__(16) int8_t sA[BN * ASTR];
    __shared__ __align__(16) int8_t sB[BM * ASTR];
    __shared__ __align__(16) float sW[NBS][BN];   // ws (q8/q4) or d*sc (Q4_K)
    __shared__ __align__(16) float sWm[NBS][BN];  // dmin*m (Q4_K)
    __shared__ float sX[NBS][BM];                 // xs
    __shared__ float sXs[NBS][BM];                // xs * block sum (Q4_K)

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr0 = (wave / WT) * RT * 32, wm0 = (wave % WT) * TT * 32;
    const int K = a.K, nb = K / BLOCK;
    // row tiles past the first weight's are the second's, then the third's
    int bx = (int)blockIdx.x;
    if (a.y2) {
        const int nx = (a.N + BN - 1) / BN, nx2 = (a.N2 + BN - 1) / BN;
        const size_t planes = a.ksplit > 1 ? (size_t)a.ksplit * a.M : 0;
        if (bx >= nx + nx2) {
            bx -= nx + nx2, a.part += planes * (size_t)(a.N + a.N2);
            a.w = a.w3, a.ws = a.ws3, a.bias = a.bias3, a.y = a.y3, a.N = a.N3;
        } else if (bx >= nx) {
            bx -= nx, a.part += planes * (size_t)a.N;
            a.w = a.w2, a.ws = a.ws2, a.bias = a.bias2, a.y = a.y2, a.N = a.N2;
            a.wtab = a.wtab2, a.wstab = a.wstab2;
        }
    }
    const int n0 = bx * BN;

    // the workgroup's rows of activations (and, grouped, its expert)
    int m0, m_end;
    const void *wp = a.w;
    const float *wsp = a.ws;
    if (a.tiles) {
        const int t = blockIdx.y;
        if (t >= a.tiles[0]) return;  // the grid is sized for the most tiles grouping can make
        const int x = a.tiles[1 + 3 * t];
        m0 = a.tiles[2 + 3 * t];
        m_end = m0 + a.tiles[3 + 3 * t];
        wp = a.wtab[x];
        wsp = a.wstab[x];
    } else {
        m0 = blockIdx.y * BM;
        m_end = a.M;
    }

    const size_t wbytes = PREC == KH_Q8 ? (size_t)a.N * K
                          : PREC == KH_Q4 ? (size_t)a.N * K / 2
                                          : (size_t)a.N * (K / QK_K) * Q4K_BYTES;
    const rsrc_t W = rsrc(wp, wbytes);
    const rsrc_t WS = rsrc(wsp, PREC == KH_Q4K ? 0 : (size_t)a.N * nb * 4);
    const rsrc_t X = rsrc(a.xq, (size_t)a.M * K);
    const rsrc_t XS = rsrc(a.xs, (size_t)a.M * nb * 4);
    const rsrc_t XSUM = rsrc(a.xsum, PREC == KH_Q4K ? (size_t)a.M * nb * 4 : 0);

    // source activation row of each of this thread's chunks (-1: none)
    int brow[B_PT], srow[XS_PT];
#pragma unroll
    for (int u = 0; u < B_PT; u++) {
        const int r = m0 + ((tid + u * THREADS) >> 3);
        brow[u] = tid + u * THREADS < B_CH && r < m_end ? (a.gather ? a.gather[r] : r) : -1;
    }
#pragma unroll
    for (int u = 0; u < XS_PT; u++) {
        const int r = m0 + (tid + u * THREADS) / NBS;
        srow[u] = tid + u * THREADS < BM * NBS && r < m_end ? (a.gather ? a.gather[r] : r) : -1;
    }

    int4 ra[A_PT], rb[B_PT], rh;
    float rws[WS_PT], rxs[XS_PT], rxsum[XS_PT];

    // Every load is issued, the ones past a tail with an offset past the
    // buffer's end, which reads zeros: no branch around any load.
    constexpr unsigned OOB = 0xffffffffu;
    auto load_stage = [&](int k0) {
#pragma unroll
        for (int u = 0; u < A_PT; u++) {
            const int c = tid + u * THREADS;
            unsigned off;
            if constexpr (PREC == KH_Q8) {
                const int row = c >> 3, kc = c & 7;
                off = c < A_CH && k0 + 16 * kc < K ? (unsigned)(n0 + row) * (unsigned)K + (unsigned)(k0 + 16 * kc) : OOB;
            } else if constexpr (PREC == KH_Q4) {
                const int row = c / NBS, blk = c % NBS;
                off = c < A_CH && k0 / BLOCK + blk < nb
                          ? (unsigned)(n0 + row) * (unsigned)(K / 2) + (unsigned)((k0 / BLOCK + blk) * 16)
                          : OOB;
            } else {
                const int row = c / NBS, q = c % NBS;
                const unsigned sb = (unsigned)(k0 / QK_K), h = (unsigned)((k0 % QK_K) / BK);
                off = c < A_CH ? (unsigned)(n0 + row) * (unsigned)(K / QK_K) * Q4K_BYTES + sb * Q4K_BYTES + 16 +
                                     64 * h + 16 * q
                               : OOB;
            }
            ra[u] = ld16(W, off);
        }
        if constexpr (PREC == KH_Q4K)
            rh = ld16(W, tid < BN ? (unsigned)(n0 + tid) * (unsigned)(K / QK_K) * Q4K_BYTES +
                                        (unsigned)(k0 / QK_K) * Q4K_BYTES
                                  : OOB);
#pragma unroll
        for (int u = 0; u < B_PT; u++) {
            const int kc = (tid + u * THREADS) & 7;
            rb[u] = ld16(X, brow[u] >= 0 && k0 + 16 * kc < K ? (unsigned)brow[u] * (unsigned)K + (unsigned)(k0 + 16 * kc)
                                                            : OOB);
        }
        if constexpr (PREC != KH_Q4K) {
#pragma unroll
            for (int u = 0; u < WS_PT; u++) {
                const int c = tid + u * THREADS;
                const int row = c / NBS, blk = c % NBS;
                rws[u] = ldf(WS, c < BN * NBS && k0 / BLOCK + blk < nb
                                     ? ((unsigned)(n0 + row) * (unsigned)nb + (unsigned)(k0 / BLOCK + blk)) * 4u
                                     : OOB);
            }
        }
#pragma unroll
        for (int u = 0; u < XS_PT; u++) {
            const int blk = (tid + u * THREADS) % NBS;
            const bool ok = srow[u] >= 0 && k0 / BLOCK + blk < nb;
            const unsigned off = ok ? ((unsigned)srow[u] * (unsigned)nb + (unsigned)(k0 / BLOCK + blk)) * 4u : OOB;
            rxs[u] = ldf(XS, off);
            if constexpr (PREC == KH_Q4K) rxsum[u] = (float)ldi(XSUM, off);
        }
    };

    auto store_stage = [&](int k0) {
#pragma unroll
        for (int u = 0; u < A_PT; u++) {
            const int c = tid + u * THREADS;
            if (c >= A_CH) continue;
            if constexpr (PREC == KH_Q8) {
                const int row = c >> 3, kc = c & 7;
                *reinterpret_cast<int4 *>(sA + row * ASTR + 16 * kc) = ra[u];
            } else if constexpr (PREC == KH_Q4) {
                // byte i of a block: weight i (low nibble), weight 16 + i (high), quant.rs:258-274
                const int row = c / NBS, blk = c % NBS;
                const int4 x = ra[u];
                int4 lo = {nib_minus8(x.x & 0x0f0f0f0f), nib_minus8(x.y & 0x0f0f0f0f), nib_minus8(x.z & 0x0f0f0f0f),
                           nib_minus8(x.w & 0x0f0f0f0f)};
                int4 hi = {nib_minus8((x.x >> 4) & 0x0f0f0f0f), nib_minus8((x.y >> 4) & 0x0f0f0f0f),
                           nib_minus8((x.z >> 4) & 0x0f0f0f0f), nib_minus8((x.w >> 4) & 0x0f0f0f0f)};
                *reinterpret_cast<int4 *>(sA + row * ASTR + 32 * blk) = lo;
                *reinterpret_cast<int4 *>(sA + row * ASTR + 32 * blk + 16) = hi;
            } else {
                // qs byte p of the super-block: sub-block 2(p/32) in the low
                // nibble, 2(p/32)+1 in the high, weight p%32 (mpp.rs:308-313)
                const int row = c / NBS, q = c % NBS;
                const int4 x = ra[u];
                int4 lo = {x.x & 0x0f0f0f0f, x.y & 0x0f0f0f0f, x.z & 0x0f0f0f0f, x.w & 0x0f0f0f0f};
                int4 hi = {(x.x >> 4) & 0x0f0f0f0f, (x.y >> 4) & 0x0f0f0f0f, (x.z >> 4) & 0x0f0f0f0f,
                           (x.w >> 4) & 0x0f0f0f0f};
                const int base = 64 * (q >> 1) + 16 * (q & 1);
                *reinterpret_cast<int4 *>(sA + row * ASTR + base) = lo;
                *reinterpret_cast<int4 *>(sA + row * ASTR + base + 32) = hi;
            }
        }
        if constexpr (PREC == KH_Q4K) {
            if (tid < BN) {
                // 6-bit scales and minimums of the stage's four sub-blocks
                // (scale_min, mpp.rs:276-282)
                const unsigned hb[4] = {(unsigned)rh.x, (unsigned)rh.y, (unsigned)rh.z, (unsigned)rh.w};
                auto byte = [&](int i) { return (hb[i >> 2] >> (8 * (i & 3))) & 0xffu; };  // block byte i
                const float d = half_bits_to_float(hb[0]), dmin = half_bits_to_float(hb[0] >> 16);
                // sub-blocks j = 4 h + jj, h the stage's half of the super-block;
                // each branch indexes the header with constants (a runtime index
                // would put it in scratch memory)
                auto put = [&](int jj, unsigned sc, unsigned mn) {
                    sW[jj][tid] = d * (float)sc;
                    sWm[jj][tid] = dmin * (float)mn;
                };
                if ((k0 % QK_K) / BK == 0) {
#pragma unroll
                    for (int j = 0; j < 4; j++) put(j, byte(4 + j) & 63, byte(8 + j) & 63);
                } else {
#pragma unroll
                    for (int j = 4; j < 8; j++)
                        put(j - 4, (byte(4 + j + 4) & 0xf) | ((byte(4 + j - 4) >> 6) << 4),
                            (byte(4 + j + 4) >> 4) | ((byte(4 + j) >> 6) << 4));
                }
            }
        }
#pragma unroll
        for (int u = 0; u < B_PT; u++) {
            const int c = tid + u * THREADS;
            if (c < B_CH) *reinterpret_cast<int4 *>(sB + (c >> 3) * ASTR + 16 * (c & 7)) = rb[u];
        }
        if constexpr (PREC != KH_Q4K) {
#pragma unroll
            for (int u = 0; u < WS_PT; u++) {
                const int c = tid + u * THREADS;
                if (c < BN * NBS) sW[c % NBS][c / NBS] = rws[u];
            }
        }
#pragma unroll
        for (int u = 0; u < XS_PT; u++) {
            const int c = tid + u * THREADS;
            if (c < BM * NBS) {
                sX[c % NBS][c / NBS] = rxs[u];
                if constexpr (PREC == KH_Q4K) sXs[c % NBS][c / NBS] = rxs[u] * rxsum[u];
            }
        }
    };

    v16f acc[RT][TT];
#pragma unroll
    for (int rt = 0; rt < RT; rt++)
#pragma unroll
        for (int tt = 0; tt < TT; tt++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[rt][tt][v] = 0.0f;

    const v16i zero = {};
    const v32f fzero32 = {};
    // One tile's products are held while the next tile's are issued: the
    // matrix core works on tile i while the VALU scales tile i - 1
    // (otherwise every convert waits out its own MFMA).  Tile s of a stage
    // (s = (b RT + rt) TT + tt) keeps its dots in D[s & 1] and its scale
    // products in half h of the pair product P, so nothing is copied
    // between steps; every index is a constant of the unrolled stage (a
    // stage holds an even number of tiles, so the tile pending at a full
    // stage's end is always D[1], half 1).
    v16i D[2] = {};
    v32f P = {};
    bool pending = false;
    auto scale_into = [&](v16f &c, const v32f &pp, int h, const v16i &d) {
#pragma unroll
        for (int v = 0; v < 16; v++) c[v] = __builtin_fmaf(pp[16 * h + v], (float)d[v], c[v]);
    };
    static_assert((NBS * RT * TT) % 2 == 0, "an even number of tiles a stage");
    // split z's stages (all of them without a split)
    int k_begin = 0, k_end = K;
    if (a.ksplit > 1) {
        const int S = (K + BK - 1) / BK, per = (S + a.ksplit - 1) / a.ksplit;
        k_begin = min(S, (int)blockIdx.z * per) * BK;
        k_end = min(K, k_begin + per * BK);
    }
    if (k_begin < k_end) load_stage(k_begin);
    for (int k0 = k_begin; k0 < k_end; k0 += BK) {
        __syncthreads();  // the previous stage's reads of LDS are done
        store_stage(k0);
        __syncthreads();
        if (k0 + BK < k_end) load_stage(k0 + BK);  // in flight during this stage's MFMAs
        const int nblk = min(NBS, (K - k0) / BLOCK);
        // block b's fragments (and its scale columns) from LDS; the next
        // block's are read while this one's products are scaled
        v4i af[2][RT], bf[2][TT];
        // The block's scale products p[r][t] = ws[r] * xs[t] (quant.rs:903;
        // Q4_K: d*sc * xs) are outer products on the matrix core, two 32 x 32
        // tiles per v_mfma_f32_32x32x1_2b_f32 (tile k from lanes 32k..32k+31
        // of both operands, its products in elements 16k..16k+15): the two
        // token tiles of a row tile (TT = 2), else the two row tiles (RT = 2),
        // else two consecutive blocks of the one tile (issued at even blocks).
        constexpr int PR = TT == 2 ? RT : 1;  // pair products per block
        float wa[2][PR], xb[2];
        auto frags = [&](int b, int f) {
#pragma unroll
            for (int rt = 0; rt < RT; rt++)
                af[f][rt] = *reinterpret_cast<const v4i *>(sA + (wr0 + rt * 32 + (lane & 31)) * ASTR + b * 32 +
                                                           16 * (lane >> 5));
#pragma unroll
            for (int tt = 0; tt < TT; tt++)
                bf[f][tt] = *reinterpret_cast<const v4i *>(sB + (wm0 + tt * 32 + (lane & 31)) * ASTR + b * 32 +
                                                           16 * (lane >> 5));
            if constexpr (TT == 2) {
#pragma unroll
                for (int rt = 0; rt < RT; rt++) wa[f][rt] = sW[b][wr0 + rt * 32 + (lane & 31)];
                xb[f] = sX[b][wm0 + lane];
            } else if constexpr (RT == 2) {
                wa[f][0] = sW[b][wr0 + lane];
                xb[f] = sX[b][wm0 + (lane & 31)];
            } else if ((b & 1) == 0) {  // blocks b and b + 1 (b + 1 < NBS: NBS is even)
                wa[f][0] = sW[b + (lane >> 5)][wr0 + (lane & 31)];
                xb[f] = sX[b + (lane >> 5)][wm0 + (lane & 31)];
            }
        };
        static_assert(NBS % 2 == 0, "block pairs stay within a stage");
        // the half of its pair product that tile (b, rt, tt) takes
        auto half_of = [](int b, int rt, int tt) { return TT == 2 ? tt : RT == 2 ? rt : b & 1; };
        frags(0, 0);
#pragma unroll
        for (int b = 0; b < NBS; b++) {
            if (b >= nblk) {  // a k tail (the last stage only): its last tile is scaled now
                const int sp = b * RT * TT - 1;
                scale_into(acc[RT - 1][TT - 1], P, half_of(b - 1, RT - 1, TT - 1), D[sp & 1]);
                pending = false;
                break;
            }
            const int f = b & 1;
#pragma unroll
            for (int rt = 0; rt < RT; rt++)
#pragma unroll
                for (int tt = 0; tt < TT; tt++) {
                    const int st = (b * RT + rt) * TT + tt;
                    D[st & 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[f][rt], bf[f][tt], zero, 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                    if (rt == 0 && tt == 0 && b + 1 < NBS && b + 1 < nblk) frags(b + 1, f ^ 1);
                    // the previous tile: (rt, tt - 1), (rt - 1, TT - 1), or the last block's last
                    const int sp = (st + 1) & 1;
                    if (tt > 0) scale_into(acc[rt][tt - 1], P, half_of(b, rt, tt - 1), D[sp]);
                    else if (rt > 0) scale_into(acc[rt - 1][TT - 1], P, half_of(b, rt - 1, TT - 1), D[sp]);
                    else if (pending) scale_into(acc[RT - 1][TT - 1], P, half_of(b - 1, RT - 1, TT - 1), D[sp]);
                    // a pair's product is issued at its first tile, once the
                    // previous pair's last half is used (one pair live at a time)
                    if (half_of(b, rt, tt) == 0) {
                        const float wv = TT == 2 ? wa[f][rt] : wa[f][0];
                        P = __builtin_amdgcn_mfma_f32_32x32x1f32(wv, xb[f], fzero32, 0, 0, 0);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    pending = true;
                }
            if constexpr (PREC == KH_Q4K) {
                // the minimum terms, sum_b dmin*m[r,b] * xs[t,b]*sum[t,b], are a
                // product over blocks: two blocks per 32x32x2 product, straight
                // into the accumulators (mpp.rs:304-315: w = d*sc*q - dmin*m)
                if (b & 1) {
                    const int bb = b - 1 + (lane >> 5);
                    float ma[RT], sb[TT];
#pragma unroll
                    for (int rt = 0; rt < RT; rt++) ma[rt] = -sWm[bb][wr0 + rt * 32 + (lane & 31)];
#pragma unroll
                    for (int tt = 0; tt < TT; tt++) sb[tt] = sXs[bb][wm0 + tt * 32 + (lane & 31)];
#pragma unroll
                    for (int rt = 0; rt < RT; rt++)
#pragma unroll
                        for (int tt = 0; tt < TT; tt++)
                            acc[rt][tt] = __builtin_amdgcn_mfma_f32_32x32x2f32(ma[rt], sb[tt], acc[rt][tt], 0, 0, 0);
                }
            }
        }
    }
    if (pending) scale_into(acc[RT - 1][TT - 1], P, 1, D[1]);
    if (a.ksplit > 1) store_partials<RT, TT>(a, acc, n0 + wr0, m0 + wm0, m_end, lane);
    else store_tiles<RT, TT>(a, acc, n0 + wr0, m0 + wm0, m_end, lane);
}

// ---------------------------------------------------------------------------
// f32 GEMM: v_mfma_f32_32x32x2_f32
// ---------------------------------------------------------------------------

constexpr int FK = 32;          // k per stage (floats)
constexpr int FSTR = FK + 4;    // LDS row stride, floats

template <int WR, int WT, int RT, int TT>
__global__ __launch_bounds__(THREADS) void gemm_f32_kernel(GemmArgs a) {
    constexpr int BN = WR * RT * 32, BM = WT * TT * 32;
    constexpr int A_CH = BN * (FK / 4), B_CH = BM * (FK / 4);
    constexpr int A_PT = (A_CH + THREADS - 1) / THREADS, B_PT = (B_CH + THREADS - 1) / THREADS;
    __shared__ __align__(16) float sA[BN * FSTR];
    __shared__ __align__(16) float sB[BM * FSTR];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr0 = (wave / WT) * RT * 32, wm0 = (wave % WT) * TT * 32;
    const int n0 = blockIdx.x * BN, m0 = blockIdx.y * BM;
    const int K = a.K;
    const rsrc_t W = rsrc(a.w, (size_t)a.N * K * 4);
    const rsrc_t X = rsrc(a.xf, (size_t)a.M * K * 4);

    int4 ra[A_PT], rb[B_PT];
    auto load_stage = [&](int k0) {
#pragma unroll
        for (int u = 0; u < A_PT; u++) {
            const int c = tid + u * THREADS, row = c / (FK / 4), kc = c % (FK / 4);
            ra[u] = c < A_CH && k0 + 4 * kc < K ? ld16(W, ((unsigned)(n0 + row) * (unsigned)K + (unsigned)(k0 + 4 * kc)) * 4u)
                                                 : int4{0, 0, 0, 0};
        }
#pragma unroll
        for (int u = 0; u < B_PT; u++) {
            const int c = tid + u * THREADS, tok = c / (FK / 4), kc = c % (FK / 4);
            rb[u] = c < B_CH && k0 + 4 * kc < K ? ld16(X, ((unsigned)(m0 + tok) * (unsigned)K + (unsigned)(k0 + 4 * kc)) * 4u)
                                                 : int4{0, 0, 0, 0};
        }
    };
    auto store_stage = [&]() {
#pragma unroll
        for (int u = 0; u < A_PT; u++) {
            const int c = tid + u * THREADS;
            if (c < A_CH) *reinterpret_cast<int4 *>(sA + (c / (FK / 4)) * FSTR + 4 * (c % (FK / 4))) = ra[u];
        }
#pragma unroll
        for (int u = 0; u < B_PT; u++) {
            const int c = tid + u * THREADS;
            if (c < B_CH) *reinterpret_cast<int4 *>(sB + (c / (FK / 4)) * FSTR + 4 * (c % (FK / 4))) = rb[u];
        }
    };

    v16f acc[RT][TT];
#pragma unroll
    for (int rt = 0; rt < RT; rt++)
#pragma unroll
        for (int tt = 0; tt < TT; tt++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[rt][tt][v] = 0.0f;

    // split z's stages (all of them without a split)
    int k_begin = 0, k_end = K;
    if (a.ksplit > 1) {
        const int S = (K + FK - 1) / FK, per = (S + a.ksplit - 1) / a.ksplit;
        k_begin = min(S, (int)blockIdx.z * per) * FK;
        k_end = min(K, k_begin + per * FK);
    }
    if (k_begin < k_end) load_stage(k_begin);
    for (int k0 = k_begin; k0 < k_end; k0 += FK) {
        __syncthreads();
        store_stage();
        __syncthreads();
        if (k0 + FK < k_end) load_stage(k0 + FK);
        // lane half h takes k = 16h + 4q + e of the stage; A and B agree on it
#pragma unroll
        for (int q = 0; q < 4; q++) {
            float4 af[RT], bf[TT];
#pragma unroll
            for (int rt = 0; rt < RT; rt++)
                af[rt] = *reinterpret_cast<const float4 *>(sA + (wr0 + rt * 32 + (lane & 31)) * FSTR +
                                                           16 * (lane >> 5) + 4 * q);
#pragma unroll
            for (int tt = 0; tt < TT; tt++)
                bf[tt] = *reinterpret_cast<const float4 *>(sB + (wm0 + tt * 32 + (lane & 31)) * FSTR +
                                                           16 * (lane >> 5) + 4 * q);
#pragma unroll
            for (int rt = 0; rt < RT; rt++)
#pragma unroll
                for (int tt = 0; tt < TT; tt++) {
                    acc[rt][tt] = __builtin_amdgcn_mfma_f32_32x32x2f32(af[rt].x, bf[tt].x, acc[rt][tt], 0, 0, 0);
                    acc[rt][tt] = __builtin_amdgcn_mfma_f32_32x32x2f32(af[rt].y, bf[tt].y, acc[rt][tt], 0, 0, 0);
                    acc[rt][tt] = __builtin_amdgcn_mfma_f32_32x32x2f32(af[rt].z, bf[tt].z, acc[rt][tt], 0, 0, 0);
                    acc[rt][tt] = __builtin_amdgcn_mfma_f32_32x32x2f32(af[rt].w, bf[tt].w, acc[rt][tt], 0, 0, 0);
                }
        }
    }
    if (a.ksplit > 1) store_partials<RT, TT>(a, acc, n0 + wr0, m0 + wm0, a.M, lane);
    else store_tiles<RT, TT>(a, acc, n0 + wr0, m0 + wm0, a.M, lane);
}

// Tile shape for a problem: the largest tile that still gives every CU a
// workgroup, else the smallest.
enum Shape { T128x128, T128x64, T128x32, T64x64 };

// The split-K workspace: one fixed allocation for the partials, made on the
// first split launch and never moved, so graphs captured over later launches
// stay valid; a split whose partials do not fit is cut to what fits, and where
// the device has no room for it nothing is split.
size_t split_bytes() { return (size_t)env_int("KVAD_GEMM_SPLIT_MIB", 64) << 20; }  // tuning knob (0: no splits)

const int SPLIT_MIN_STAGES = env_int("KVAD_GEMM_SPLIT_MIN", 2);  // tuning knobs
const int SPLIT_MAX = env_int("KVAD_GEMM_SPLIT_MAX", 32);
const int SPLIT_PER_CU = env_int("KVAD_GEMM_SPLIT_PER_CU", 2);
// Under twelve stages of 128 a second launch costs more than two shorter chains
// save ((512 tokens, 896 rows, 896) 14.1 us in two splits, 11.2 unsplit, (80,
// 4864, 896) 14.0 and 10.9), and so do a joint launch's two or three; three chains
// and more of one weight pay for it (Q4_K (90, 1968, 1280) 19.2 us unsplit, 12.7
// in five, (85, 3146, 1280) 20.1 and 17.0 in three; q8 (72, 96, 1376) 13.6 and
// 10.3).
constexpr int SPLIT_LEAST = 12;

// Rows of every weight of a launch, and their tiles.
long long all_rows(const GemmArgs &a) { return (long long)a.N + (a.y2 ? a.N2 : 0) + (a.y3 ? a.N3 : 0); }
long long row_tiles(const GemmArgs &a, int tile_n) {
    auto tiles = [&](int n) { return ((long long)n + tile_n - 1) / tile_n; };
    return tiles(a.N) + (a.y2 ? tiles(a.N2) : 0) + (a.y3 ? tiles(a.N3) : 0);
}

bool rows_in_fours(const GemmArgs &a) { return !(a.N % 4 || (a.y2 && a.N2 % 4) || (a.y3 && a.N3 % 4)); }

// How many splits a launch's k-stages are cut into (under 2: none): `stages` of
// them, at least `min_st` a split, under `least` three splits or none, so that the grid comes to
// about SPLIT_PER_CU workgroups per CU (a CU holds several: one's loads wait while
// another's MFMAs run), at most SPLIT_MAX splits, and partials (4 M N bytes a
// split, written and read again) of at most the weights' wbytes or 4 MiB,
// whichever is more (a small weight such as a router's 64 rows would otherwise
// never split: 512 tokens x 64 x 2048, 16 workgroups, 22.6 us unsplit).  Up to
// `twice` splits (128 x 128 tiles, which fill a round by them, and f32: any; else
// four) may take twice that from `least` + 4 stages on, where the tiles fill half
// the CUs or fewer and the rows are in fours ((512 tokens, 1024 rows, 4096) 25.2 ->
// 22.7 us in four splits instead of two, Q4_K 36.7 -> 28.2, (512, 896, 4864) 27.2 ->
// 24.9; (512, 2048, 2048), a tile for every CU, 19.0 unsplit, 24.9 in two); more
// than four do not pay for it ((128, 896, 4864) in nine 14.6, in eighteen 15.6),
// nor do rows whose partials go value by value (q8 (313, 477, 4544) 21.5 and 26.9).
long long split_count(const GemmArgs &a, long long tiles, int stages, int min_st, int least, int twice, size_t wbytes,
                      int cu) {
    const size_t plane = (size_t)a.M * all_rows(a) * 4;
    const size_t most = std::max(wbytes, (size_t)4 << 20);
    long long most_ks = (long long)(most / plane);
    if (most_ks < twice && stages >= least + 4 && 2 * tiles <= cu && rows_in_fours(a))
        most_ks = std::min<long long>(twice, (long long)(2 * most / plane));
    long long ks = ((long long)SPLIT_PER_CU * cu + tiles / 2) / tiles;
    ks = std::min<long long>(ks, stages / min_st);
    ks = std::min<long long>(ks, SPLIT_MAX);
    ks = std::min<long long>(ks, most_ks);
    if (stages < least && (ks < 3 || a.y2)) ks = 1;
    const int forced = env_int("KVAD_GEMM_KSPLIT", 0);  // tuning knob: k splits (1: none)
    if (forced > 0) ks = std::min(forced, stages);
    return std::min<long long>(ks, (long long)(split_bytes() / plane));
}
// The int8 GEMM's, in tiles of tile_m tokens by tile_n rows.
long long split_count_i8(const GemmArgs &a, int tile_m, int tile_n, int cu) {
    return split_count(a, row_tiles(a, tile_n) * ((a.M + tile_m - 1) / tile_m), (a.K + BK - 1) / BK, SPLIT_MIN_STAGES,
                       SPLIT_LEAST, tile_m == 128 ? SPLIT_MAX : 4, (size_t)all_rows(a) * a.K, cu);
}

// Whether 128 x 128 tiles, of which a CU holds two, use the chip well enough
// over rows long enough to pay for a workgroup's start.  They need half
// the LDS and scale traffic of 64 x 64 tiles, but a round that is short of
// workgroups costs a whole one: taken from seven eighths of a round of two a CU,
// and from a round and a half on, where the sweep had them ahead whether the last
// one is full or not.  Measured (us, rows' quantisation included, 64 x
// 64 tiles / 128 x 128): Q4_K 14336x4096 at 512 / 700 / 1000 tokens, 448 / 672 /
// 896 tiles, 157 / 210 / 282 and 138 / 226 / 268; q8 115 / 160 / 221 and 107 / 165 /
// 208; 8192x2048 at 700 / 1000 / 1500, 384 / 512 / 768 tiles, 53 / 70 / 99 and 60 /
// 63 / 92; q8 9728x896 at 700, 456 tiles of seven stages, 32.5 and 33.5.  Fewer
// tiles fill a round split along k, from 13 stages a split of 8192 columns or
// more: 4096x14336 at 256 / 384 / 512 / 700 / 1000 tokens, 512 / 480 / 512 / 576 / 512
// workgroups, Q4_K 107 / 189 / 189 / 225 / 353 and 80 / 116 / 141 / 273 / 266, q8 75 /
// 124 / 130 / 164 / 231 and 65 / 93 / 112 / 202 / 206; shorter
// splits go both ways (4096x4096 at 512 tokens, eight stages, 43.6 and 47.9,
// 2048x8192 at 700, 12.8, 76 and 64).  Token tiles more than an
// eighth empty are left to the smaller ones, and so are six splits and more of
// q8 and q4 rows that are no multiple of four, whose partials go value by value
// (574 tokens, 1082 rows, 18528 columns, eleven splits, 76 and 112; 586, 1152,
// 18688, eleven, 82 and 74; over 24 shapes of six to eleven splits 0.68 to 1.01 of
// the smaller tiles' speed, of rows in fours 0.96 to 1.27; Q4_K 0.93 to 1.48 over
// either).
bool fills_rounds(kh_ctx *ctx, int precision, const GemmArgs &a, long long cu) {
    const long long M = a.M, mt = (M + 127) / 128, t = row_tiles(a, 128) * mt, stages = (a.K + BK - 1) / BK;
    if (M < 128 || 8 * 128 * mt > 9 * M) return false;
    if (t > cu) return stages >= 16 && (t >= 3 * cu || (4 * t >= 7 * cu && t <= 2 * cu));
    if (stages < 64) return false;
    const long long ks = split_count_i8(a, 128, 128, (int)cu);
    if (ks > 5 && !rows_in_fours(a) && precision != KH_Q4K) return false;
    return ks >= 2 && stages >= 13 * ks && 4 * t * ks >= 7 * cu && t * ks <= 2 * cu && split_partials(ctx, 0);
}
Shape pick_shape(kh_ctx *ctx, int precision, const GemmArgs &a) {
    const int forced = env_int("KVAD_GEMM_TILE_M", 0);  // tuning knob: tokens per tile (6464: 64 x 64)
    if (forced == 6464) return T64x64;
    if (forced == 128 || forced == 64 || forced == 32) return forced == 128 ? T128x128 : forced == 64 ? T128x64 : T128x32;
    const int cu = ctx->cu_count > 0 ? ctx->cu_count : 256, M = a.M;
    const long long nt = row_tiles(a, 128);
    // 128 x 128 tiles while they give four workgroups per CU, or fill their
    // rounds of the chip; else, past 64 tokens, 64 x 64 tiles: more, smaller workgroups hide the k-stages' load
    // latency ((512, 896, 4864) 28.5 -> 27.4 us against 128-row 32-token tiles,
    // (512, 4864, 896) 19.1 -> 17.8, (128, 896, 896) 10.9 -> 10.3, all split alike;
    // at (2048, 4096, 14336) they lose, 461 -> 597, and at 16 tokens over
    // 14336x4096 29 -> 45 against 32-token tiles split over k).
    // Token tiles no wider than the tokens need: a tall matrix at 16 or 32
    // tokens (a vocabulary head) gives enough workgroups with 32-token
    // tiles, and 128-token ones would leave three quarters of every tile idle.
    if (M > 64 && nt * ((M + 127) / 128) >= 4LL * cu) return T128x128;
    if (fills_rounds(ctx, precision, a, cu)) return T128x128;
    if (M > 64 && M < 128 && nt >= cu) return T128x128;
    // three token tiles of 32 rather than two of 64, half of the second empty:
    // Q4_K, whose tiles cost the most (67 tokens, 5728 rows, 12544 columns 77 -> 66
    // us, (80, 3028, 6144) 27.0 -> 24.6); q8 and q4 are behind over small weights
    // (q8 (68, 2196, 3456) 14.8 -> 16.6)
    if (M > 64 && M <= 96 && precision == KH_Q4K) return T128x32;
    if (M > 64) return T64x64;
    if (M > 32 && nt >= cu) return T128x64;
    return T128x32;
}

}  // namespace

int gemm_tiles(kh_ctx *ctx, int precision, const GemmArgs &a, int *tile_n) {
    const Shape sh = pick_shape(ctx, precision, a);
    *tile_n = sh == T64x64 ? 64 : 128;
    return sh == T128x128 ? 128 : sh == T128x32 ? 32 : 64;
}

namespace {

template <int PREC>
int launch_i8(kh_ctx *ctx, const GemmArgs &a, int max_tiles, int tile_m, int tile_n) {
    const unsigned gx = (unsigned)row_tiles(a, tile_n);
    const unsigned gy = a.tiles ? (unsigned)max_tiles : (unsigned)((a.M + tile_m - 1) / tile_m);
    if (gy == 0) return KH_OK;
    const dim3 grid(gx, gy, a.ksplit > 1 ? (unsigned)a.ksplit : 1u);
    if (tile_n == 64) {
        if (tile_m != 64 || a.tiles) return fail(KH_EINVAL, "gemm: 64-row tiles are 64 tokens wide and ungrouped");
        hipLaunchKernelGGL((gemm_i8_kernel<PREC, 2, 2, 1, 1>), grid, dim3(THREADS), 0, ctx->stream, a);
    } else switch (tile_m) {
        case 128:
            hipLaunchKernelGGL((gemm_i8_kernel<PREC, 2, 2, 2, 2>), grid, dim3(THREADS), 0, ctx->stream, a);
            break;
        case 64:
            hipLaunchKernelGGL((gemm_i8_kernel<PREC, 2, 2, 2, 1>), grid, dim3(THREADS), 0, ctx->stream, a);
            break;
        default:
            hipLaunchKernelGGL((gemm_i8_kernel<PREC, 4, 1, 1, 1>), grid, dim3(THREADS), 0, ctx->stream, a);
            break;
    }
    KH_HIP(hipGetLastError());
    if (a.ksplit > 1) {
        const int ns[3] = {a.N, a.y2 ? a.N2 : 0, a.y3 ? a.N3 : 0};
        const float *bias[3] = {a.bias, a.bias2, a.bias3};
        float *y[3] = {a.y, a.y2, a.y3};
        const float *part = a.part;
        for (int i = 0; i < 3 && ns[i]; i++) {
            const int rc = launch_split_reduce(ctx, part, a.ksplit, a.M, ns[i], bias[i], a.accumulate, y[i]);
            if (rc) return rc;
            part += (size_t)a.ksplit * a.M * ns[i];
        }
    }
    return KH_OK;
}

void plan_split_f32(kh_ctx *ctx, GemmArgs &a, int tile_m);

// The f32 GEMM runs best on shorter token tiles than the int8 one (swept at
// both prefill shapes): 64 tokens while that still gives two workgroups per
// CU, else 32.
Shape pick_shape_f32(int M, int N, int cu) {
    const int forced = env_int("KVAD_GEMM_TILE_M", 0);
    if (forced == 128 || forced == 64 || forced == 32) return forced == 128 ? T128x128 : forced == 64 ? T128x64 : T128x32;
    const long long nt = (N + 127) / 128;
    return nt * ((M + 63) / 64) >= 2LL * cu ? T128x64 : T128x32;
}

int launch_f32gemm(kh_ctx *ctx, GemmArgs a) {
    const int cu = ctx->cu_count > 0 ? ctx->cu_count : 256;
    const Shape sh = pick_shape_f32(a.M, a.N, cu);
    const int tile_m = sh == T128x128 ? 128 : sh == T128x64 ? 64 : 32;
    plan_split_f32(ctx, a, tile_m);
    const dim3 grid((unsigned)((a.N + 127) / 128), (unsigned)((a.M + tile_m - 1) / tile_m),
                    a.ksplit > 1 ? (unsigned)a.ksplit : 1u);
    switch (sh) {
        case T128x128:
            hipLaunchKernelGGL((gemm_f32_kernel<2, 2, 2, 2>), grid, dim3(THREADS), 0, ctx->stream, a);
            break;
        case T128x64:
            hipLaunchKernelGGL((gemm_f32_kernel<2, 2, 2, 1>), grid, dim3(THREADS), 0, ctx->stream, a);
            break;
        default:
            hipLaunchKernelGGL((gemm_f32_kernel<4, 1, 1, 1>), grid, dim3(THREADS), 0, ctx->stream, a);
            break;
    }
    KH_HIP(hipGetLastError());
    if (a.ksplit > 1) return launch_split_reduce(ctx, a.part, a.ksplit, a.M, a.N, a.bias, a.accumulate, a.y);
    return KH_OK;
}

// Row-at-a-time path for shapes the tiled kernels do not take (f32 weights
// whose width is not a multiple of 4): one GEMV job per activation row.
int matmul_rows(kh_ctx *ctx, const kh_weight *w, const float *xs, size_t m, const float *bias, float *y,
                int accumulate) {
    std::vector<GemvJob> jobs(m);
    for (size_t i = 0; i < m; i++) {
        GemvJob &j = jobs[i];
        j = GemvJob{};
        j.w = w->qs;
        j.xf = xs + i * w->cols;
        j.bias = bias;
        j.y = y + i * w->rows;
        j.rows = (int)w->rows;
        j.cols = (int)w->cols;
        j.accumulate = accumulate;
    }
    return launch_gemv(ctx, w->precision, jobs.data(), (int)m);
}

}  // namespace

namespace {
// KVAD_MATMUL_GEMM=1 sends every m > 1 to the MFMA GEMM (for comparisons).
bool matmul_force_gemm() { return env_int("KVAD_MATMUL_GEMM", 0) == 1; }
}  // namespace

void gemm_split_reserve(kh_ctx *ctx) {
    if (ctx->gemm.ptr || !split_bytes()) return;
    if (hipMalloc(&ctx->gemm.ptr, split_bytes()) == hipSuccess) {
        ctx->gemm.bytes = split_bytes();
    } else {
        ctx->gemm.ptr = nullptr;
        (void)hipGetLastError();  // the unsplit launch's check must not find it
    }
}

float *split_partials(kh_ctx *ctx, size_t bytes) {
    if (!ctx->gemm.ptr) {
        if (capturing(ctx->stream)) return nullptr;
        gemm_split_reserve(ctx);
    }
    return bytes <= ctx->gemm.bytes ? static_cast<float *>(ctx->gemm.ptr) : nullptr;
}

int launch_split_reduce(kh_ctx *ctx, const float *part, int ks, int M, int N, const float *bias, int accumulate,
                        float *y) {
    const size_t quads = ((size_t)M * N + 3) / 4;
    hipLaunchKernelGGL(split_reduce_kernel, dim3((unsigned)((quads + 255) / 256)), dim3(256), 0, ctx->stream, part, ks,
                       M, N, bias, accumulate, y);
    KH_HIP(hipGetLastError());
    return KH_OK;
}

namespace {

// Sets a's split-K fields for ks splits, none under two or without a workspace.
void set_split(kh_ctx *ctx, GemmArgs &a, long long ks) {
    a.ksplit = 0;
    if (ks < 2) return;
    a.part = split_partials(ctx, (size_t)ks * a.M * all_rows(a) * 4);
    if (a.part) a.ksplit = (int)ks;
}

// The f32 GEMM's split, at least two stages of 32 k-values each.  A few
// 128-row tiles over long rows had left most CUs idle and every workgroup
// waiting out its stages in turn: (90 tokens, 3000 rows, 2052 columns), 72
// workgroups of 65 stages, 56 -> 22 us; 4096x4096 at 2 / 32 / 128 tokens 114 ->
// 20 / 21 / 50; a 64x2048 router at 4 / 512 54 -> 6.3 / 10.8; 896x4864 at 16
// 126 -> 11.5; 512x512 at 16 15.7 -> 6.9 (at least four stages 8.5, eight 11.7).
void plan_split_f32(kh_ctx *ctx, GemmArgs &a, int tile_m) {
    const long long tiles = (long long)((a.N + 127) / 128) * ((a.M + tile_m - 1) / tile_m);
    const int cu = ctx->cu_count > 0 ? ctx->cu_count : 256;
    set_split(ctx, a, split_count(a, tiles, (a.K + FK - 1) / FK, 2, 0, SPLIT_MAX, (size_t)a.N * a.K * 4, cu));
}

}  // namespace

void plan_split(kh_ctx *ctx, GemmArgs &a, int tile_m, int tile_n) {
    a.ksplit = 0;
    if (a.tiles) return;  // grouped launches are not split
    set_split(ctx, a, split_count_i8(a, tile_m, tile_n, ctx->cu_count > 0 ? ctx->cu_count : 256));
}

int launch_matmul(kh_ctx *ctx, const kh_weight *w, const float *xs, size_t m, const float *bias, float *y,
                  int accumulate) {
    const size_t rows = w->rows, cols = w->cols;
    // 32-bit buffer offsets: the weights and activations (plus one tile of
    // overhang) must stay below 4 GiB
    const size_t wb = w->precision == KH_F32 ? 4 * rows * cols : rows * cols;
    const size_t xb = w->precision == KH_F32 ? 4 * m * cols : m * cols;
    if (wb + 4 * 128 * cols >= 0xffffffffull || xb + 4 * 128 * cols >= 0xffffffffull || rows > 0x7fffffff ||
        m > 0x7fffffff)
        return fail(KH_DECLINED, "matmul: operands of 4 GiB or more are not addressed here");
    GemmArgs a{};
    a.w = w->qs;
    a.ws = w->scales;
    a.bias = bias;
    a.y = y;
    a.accumulate = accumulate;
    a.M = (int)m;
    a.N = (int)rows;
    a.K = (int)cols;
    if (w->precision == KH_F32) {
        if (cols % 4) return matmul_rows(ctx, w, xs, m, bias, y, accumulate);
        a.xf = xs;
        return launch_f32gemm(ctx, a);
    }
    // a few rows: the VALU multi-token GEMV quantises them as it stages them
    // (QActBatch::new's codes, one launch fewer) while they are few values
    const bool multi = matmul_takes_multi(w->precision, m, rows, cols) && !matmul_force_gemm();
    if (multi && multi_stages_f32(w->precision, m, rows, cols))
        return launch_gemv_multi_jobs(ctx, 1, &w, &bias, &y, &accumulate, QAct{}, m, xs);
    // QActBatch::new (quant.rs:693-714): the activation rows quantised per block
    const size_t qb = (m * cols + 255) / 256 * 256, sb = (4 * m * cols / BLOCK + 255) / 256 * 256;
    int rc = ensure(ctx, ctx->ws, qb + 2 * sb);
    if (rc) return rc;
    char *p = static_cast<char *>(ctx->ws.ptr);
    QAct q{reinterpret_cast<int8_t *>(p), reinterpret_cast<float *>(p + qb), reinterpret_cast<int32_t *>(p + qb + sb)};
    if ((rc = launch_qact(ctx, xs, m, cols, q))) return rc;
    return launch_matmul_q(ctx, w, q, m, bias, y, accumulate);
}

int launch_matmul_q(kh_ctx *ctx, const kh_weight *w, const QAct &q, size_t m, const float *bias, float *y,
                    int accumulate) {
    const size_t rows = w->rows, cols = w->cols;
    if (w->precision == KH_F32) return fail(KH_EINVAL, "matmul: f32 weights take f32 rows");
    if (rows * cols + 4 * 128 * cols >= 0xffffffffull || m * cols + 4 * 128 * cols >= 0xffffffffull ||
        rows > 0x7fffffff || m > 0x7fffffff)
        return fail(KH_DECLINED, "matmul: operands of 4 GiB or more are not addressed here");
    // a few tokens: stream the weights once through the multi-token GEMV
    if (matmul_takes_multi(w->precision, m, rows, cols) && !matmul_force_gemm())
        return launch_gemv_multi_jobs(ctx, 1, &w, &bias, &y, &accumulate, q, m);
    GemmArgs a{};
    a.w = w->qs;
    a.ws = w->scales;
    a.bias = bias;
    a.y = y;
    a.accumulate = accumulate;
    a.M = (int)m;
    a.N = (int)rows;
    a.K = (int)cols;
    a.xq = q.qs;
    a.xs = q.scales;
    a.xsum = q.sums;
    int tile_n;
    const int tile_m = gemm_tiles(ctx, w->precision, a, &tile_n);
    plan_split(ctx, a, tile_m, tile_n);
    return launch_gemm_q(ctx, w->precision, a, 0, tile_m, tile_n);
}

int launch_gemm_q(kh_ctx *ctx, int precision, const GemmArgs &a, int max_tiles, int tile_m, int tile_n) {
    if (a.tiles && (!a.wtab || !a.wstab)) return fail(KH_EINVAL, "gemm: grouped launch without weight tables");
    switch (precision) {
        case KH_Q8: return launch_i8<KH_Q8>(ctx, a, max_tiles, tile_m, tile_n);
        case KH_Q4: return launch_i8<KH_Q4>(ctx, a, max_tiles, tile_m, tile_n);
        case KH_Q4K: return launch_i8<KH_Q4K>(ctx, a, max_tiles, tile_m, tile_n);
        default: return fail(KH_EINVAL, "gemm: the grouped kernel takes quantised weights");
    }
}

int launch_matmul_jobs(kh_ctx *ctx, int k, const kh_weight *const *w, const QAct &q, size_t m,
                       const float *const *bias, float *const *y) {
    if (k < 2 || k > 3) return fail(KH_EINVAL, "matmul: two or three weights per launch");
    const size_t cols = w[0]->cols;
    size_t rows = 0;
    for (int i = 0; i < k; i++) {
        if (w[i]->precision == KH_F32 || w[i]->precision != w[0]->precision || w[i]->cols != cols)
            return fail(KH_EINVAL, "matmul: weights of one launch share a quantised precision and width");
        if (w[i]->rows * cols + 4 * 128 * cols >= 0xffffffffull)
            return fail(KH_DECLINED, "matmul: operands of 4 GiB or more are not addressed here");
        rows += w[i]->rows;
    }
    if (m * cols + 4 * 128 * cols >= 0xffffffffull || rows > 0x7fffffff || m > 0x7fffffff)
        return fail(KH_DECLINED, "matmul: operands of 4 GiB or more are not addressed here");
    GemmArgs a{};
    a.M = (int)m, a.K = (int)cols;
    a.xq = q.qs, a.xs = q.scales, a.xsum = q.sums;
    a.w = w[0]->qs, a.ws = w[0]->scales, a.bias = bias[0], a.y = y[0], a.N = (int)w[0]->rows;
    a.w2 = w[1]->qs, a.ws2 = w[1]->scales, a.bias2 = bias[1], a.y2 = y[1], a.N2 = (int)w[1]->rows;
    if (k == 3) a.w3 = w[2]->qs, a.ws3 = w[2]->scales, a.bias3 = bias[2], a.y3 = y[2], a.N3 = (int)w[2]->rows;
    int tn;
    const int tm = gemm_tiles(ctx, w[0]->precision, a, &tn);
    plan_split(ctx, a, tm, tn);
    return launch_gemm_q(ctx, w[0]->precision, a, 0, tm, tn);
}

}  // namespace kh
