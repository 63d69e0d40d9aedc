// Multi-row matmul for the batched prefill: out[m, n] (+)= in[m, :] . W[n, :].
// The integer path (Q8_0 activations) runs on the matrix cores from operands
// in fragment order (gemm_tile_kernel, gemm_rows_kernel below); gemm_kernel,
// described next, serves f32 activations.
//
// A tile of MT activation rows is staged in LDS once; each wavefront then
// streams weight rows (lane = 32-block, as in the decode matvec) and dots
// every row of the tile against them, so weights are read ceil(M/MT) times
// instead of M times (the reference re-streams them per row,
// src/kernels/matmul.rs:34).
#include <atomic>
#include <cstring>

#include "launch.h"

namespace sq {
namespace {

constexpr int kPad = 36;
constexpr int WAVES = 4;
constexpr int RPW = 4;               // weight rows per wavefront
constexpr int TN = WAVES * RPW;      // weight rows per workgroup

template <int WT>
struct Dw;
template <> struct Dw<WT_Q8_0> { static constexpr int v = 8; };
template <> struct Dw<WT_Q4_0> { static constexpr int v = 4; };
template <> struct Dw<WT_BF16> { static constexpr int v = 16; };

template <int WT, int NBL, int MT>
__global__ __launch_bounds__(WAVES * 64) void gemm_kernel(MatView w, const float* __restrict__ x, int m_rows,
                                                           float* __restrict__ out, int ldo,
                                                           int accumulate) {
    constexpr int KMAX = NBL * 64 * 32;
    constexpr int DW = Dw<WT>::v;
    __shared__ __attribute__((aligned(16))) float s_x[MT * (KMAX / 32) * kPad];

    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int K = w.k, KB = K >> 5;
    const int m0 = blockIdx.y * MT;
    const int mt = min(MT, m_rows - m0);

    for (int e = tid; e < MT * K; e += WAVES * 64) {
        const int m = e / K, i = e % K;
        s_x[m * (KMAX / 32) * kPad + (i >> 5) * kPad + (i & 31)] = (m < mt) ? x[(size_t)(m0 + m) * K + i] : 0.0f;
    }
    __syncthreads();

    const uint8_t* wbase = (const uint8_t*)w.qs;
    const size_t row_bytes = (size_t)KB * DW * 4;
    for (int r = 0; r < RPW; r++) {
        const int n = blockIdx.x * TN + wave * RPW + r;
        if (n >= w.rows) break;
        int W[NBL][DW];
        float sw[NBL];
#pragma unroll
        for (int b = 0; b < NBL; b++) {
            const int blk = lane + 64 * b;
            if (blk < KB) {
                const sq_v4i* p = (const sq_v4i*)(wbase + (size_t)n * row_bytes + (size_t)blk * DW * 4);
#pragma unroll
                for (int v = 0; v < DW / 4; v++) {
                    sq_v4i t = p[v];
                    W[b][4 * v] = t.x; W[b][4 * v + 1] = t.y; W[b][4 * v + 2] = t.z; W[b][4 * v + 3] = t.w;
                }
                sw[b] = (WT == WT_BF16) ? 1.0f : sq_f16_to_f32(w.scale[(size_t)n * KB + blk]);
            } else {
#pragma unroll
                for (int v = 0; v < DW; v++) W[b][v] = 0;
                sw[b] = 0.0f;
            }
        }
        float acc[MT];
#pragma unroll
        for (int m = 0; m < MT; m++) acc[m] = 0.0f;
#pragma unroll
        for (int b = 0; b < NBL; b++) {
            const int blk = lane + 64 * b;
            if (blk >= KB) continue;
#pragma unroll
            for (int m = 0; m < MT; m++) {
                const float* xb = s_x + m * (KMAX / 32) * kPad + blk * kPad;
                float bacc = 0.0f;
                if constexpr (WT == WT_Q8_0) {
#pragma unroll
                    for (int v = 0; v < 8; v++) {
                        float4 x4 = *(const float4*)(xb + 4 * v);
                        bacc += x4.x * sq_sbyte_f(W[b][v], 0);
                        bacc += x4.y * sq_sbyte_f(W[b][v], 1);
                        bacc += x4.z * sq_sbyte_f(W[b][v], 2);
                        bacc += x4.w * sq_sbyte_f(W[b][v], 3);
                    }
                    acc[m] += bacc * sw[b];
                } else if constexpr (WT == WT_Q4_0) {
#pragma unroll
                    for (int v = 0; v < 4; v++) {
                        const unsigned dw = (unsigned)W[b][v];
                        float4 xl = *(const float4*)(xb + 4 * v);
                        float4 xh = *(const float4*)(xb + 16 + 4 * v);
                        bacc += xl.x * (float)((int)(dw & 15u) - 8) + xh.x * (float)((int)((dw >> 4) & 15u) - 8);
                        bacc += xl.y * (float)((int)((dw >> 8) & 15u) - 8) + xh.y * (float)((int)((dw >> 12) & 15u) - 8);
                        bacc += xl.z * (float)((int)((dw >> 16) & 15u) - 8) + xh.z * (float)((int)((dw >> 20) & 15u) - 8);
                        bacc += xl.w * (float)((int)((dw >> 24) & 15u) - 8) + xh.w * (float)((int)((dw >> 28) & 15u) - 8);
                    }
                    acc[m] += bacc * sw[b];
                } else {
#pragma unroll
                    for (int v = 0; v < 16; v++) {
                        const unsigned dw = (unsigned)W[b][v];
                        float2 x2 = *(const float2*)(xb + 2 * v);
                        bacc += x2.x * __builtin_bit_cast(float, dw << 16);
                        bacc += x2.y * __builtin_bit_cast(float, dw & 0xFFFF0000u);
                    }
                    acc[m] += bacc;
                }
            }
        }
#pragma unroll
        for (int m = 0; m < MT; m++) {
            const float v = sq_wave_sum(acc[m]);
            if (lane == m && m < mt) {
                float* o = out + (size_t)(m0 + m) * ldo + n;
                if (accumulate) *o += v;
                else *o = v;
            }
        }
    }
}

// ---- integer path on the matrix cores ------------------------------------------
// out[m, n] (+)= sum over blocks b of f32(isum_b[m, n]) * (sa[m, b] * sw[n, b]),
// each term fused into the running sum as the reference's aarch64 kernels
// combine blocks (dot_prod.rs:189-252; the scalar twin, dot_prod.rs:376-403,
// rounds (f32(isum) * sa) * sw instead): isum_b is the exact i32 dot of one
// 32-element block, which is one v_mfma_i32_32x32x32_i8 (the full int8 rate of
// gfx950) for a 32 x 32 tile of outputs: lane l supplies 16 bytes of row
// l % 32, half l / 32 of the block, and the other operand alike.
//
// The scale product sa * sw of two f16 values has at most 22 significant bits,
// so it is exact in f32 however it is formed; it comes from one
// v_mfma_f32_32x32x8_f16 per tile and block, already in the result layout:
// lanes 0-31 hold the block's scale of row (column) l % 32 in k-slot 0 or 1,
// zeros elsewhere.  Result element r of lane l is row 8 (r / 4) + 4 (l / 32) +
// r % 4, column l % 32.  Each element and block then takes two VALU operations.
typedef float sq_v4f __attribute__((ext_vector_type(4)));
typedef int m8_v16i __attribute__((ext_vector_type(16)));
typedef float m8_v16f __attribute__((ext_vector_type(16)));

// The block sums reach f32 without a conversion instruction: the integer
// products accumulate onto kIsumBase, the bit pattern of 1.5 * 2^23, so a
// result's bits read as the f32 1.5 * 2^23 + isum (exact for |isum| < 2^22;
// a block's sum is at most 32 * 127 * 128), and one subtraction leaves
// f32(isum), exactly.  v_cvt_f32_i32 issues at half the rate of a subtraction
// (2.4 against 1.3 ns per wavefront instruction and SIMD), and with it a
// 32 x 32 tile and block takes 50 ns per SIMD in registers alone, against 41 ns
// (two wavefronts of four tiles a SIMD, launches of 2.6 ms; 57 and 47 in
// launches of 0.2 ms; three wavefronts: 59 and 43).
// The base operand sits in registers, behind an empty asm so that the compiler
// does not set it anew for every product.
constexpr int kIsumBase = 0x4B400000;
__device__ __forceinline__ float isum_f32(int d) { return __builtin_bit_cast(float, d) - 12582912.0f; }
template <typename V>
__device__ __forceinline__ V isum_base() {
    V v;
#pragma unroll
    for (int r = 0; r < (int)(sizeof(V) / 4); r++) v[r] = kIsumBase;
    asm volatile("" : "+v"(v));
    return v;
}
typedef _Float16 mq_v4h __attribute__((ext_vector_type(4)));

// Matmul epilogues: RW_STORE writes (or adds) the tile; RW_GATEUP and RW_QKV
// are described with the kernels that take them.
enum : int { RW_STORE = 0, RW_GATEUP = 1, RW_QKV = 2, RW_SHARED = 3 };
struct FragMat {  // a matrix in fragment order
    const int8_t* q;
    const uint16_t* s;
    int rows, k;
};
// RW_SHARED (the few-rows kernel): further matrices that take the same input;
// workgroups from begin[i] on multiply w[i], storing to out[i].
struct SharedMats {
    FragMat w[kSharedMax - 1];
    float* out[kSharedMax - 1];
    int begin[kSharedMax - 1];
};
struct RowsEpi {
    int8_t* act_q;       // RW_GATEUP: FFN activation blocks [m][ffn], scales [m][ffn / 32]
    uint16_t* act_d;
    const float2* rope;  // RW_QKV: (cos, sin) per position and pair
    float* q_out;        // [m][q_dim]
    float* kcache;       // [position][kv_dim]
    float* vcache;
    int q_dim, kv_dim, head_dim, pos0;
};
// One lane's dword of packed Q4_0 nibbles (fragment order, q - 8) as four
// signed bytes of 16 (q - 8): the low nibbles for half 0 of the block (sh 4),
// the high ones for half 1 (sh 0).  Two operations a dword; the factor 16 is
// taken out of the finished sums, exactly (a power of two).
__device__ __forceinline__ sq_v4i q4_bytes(sq_v4i v, int sh) {
#pragma unroll
    for (int i = 0; i < 4; i++) v[i] = (int)(((unsigned)v[i] << sh) & 0xF0F0F0F0u);
    return v;
}
template <int WT>
constexpr float kOutScale = WT == WT_Q4_0 ? 1.0f / 16.0f : 1.0f;

// ---- the tile kernel -----------------------------------------------------------
// A wavefront computes SM x SN tiles of 32 x 32, WM x WN wavefronts a
// workgroup.  Its operands come straight from global memory into registers,
// each load 1 KB in one piece (fragment order, sq_common.h), D blocks ahead,
// with no LDS and no barrier; the wavefronts of a workgroup share rows and
// columns through the L1 cache.  Row-order operands staged through LDS with
// direct loads had been bound by those loads: 64-byte pieces, and a request
// per row and block pair for the scales (half of all L2 requests).  The gate/up
// projection of 2048 rows (16384 x 2048, Q8_0) took 185 us that way, alone, and
// takes 137 here (1005 TOP/s); of 320 rows 62, and 35-41 here.
//
// blockIdx.z: the K split [kb_begin, kb_end) of blocks, kbs (even) each; its
// tiles go to partial buffers split_stride floats apart.
//
// Epilogues: RW_GATEUP (SN = 2) takes the stacked [gate; up] matrix, a
// wavefront's two column tiles being gate rows 32 g .. and the up rows
// ffn + 32 g .., so every output element of its gate tile has its up value at
// the same register of the other tile; SiLU(gate) * up passes through LDS
// (each wavefront its own rows) and a lane takes one prompt row's FFN block:
// maximum, Q8_0 scale and quants as silu_mul8_kernel forms them.  RW_QKV
// applies RoPE to the q and k columns (the pair partner of column n is column
// n ^ 1, lane l ^ 1) and appends the K and V rows to the cache, as
// rope_kv_kernel does.  The same operations on the same values as the separate
// kernels, so the same bits.
// `base` (the same on every lane) plus a lane's byte offset.  The offset is
// opaque here, so that the address stays a scalar base and a 32-bit lane offset:
// folded into the loop-invariant part, every tile's 64-bit address would live in
// vector registers (and spill).
__device__ __forceinline__ const void* lane_at(const void* base, uint32_t off) {
    asm volatile("" : "+v"(off));
    return (const int8_t*)base + off;
}

template <int WT, int SM, int SN, int WM, int WN, int D, int EPI>
__global__ __launch_bounds__(64 * WM * WN, D == 4 ? 2 : 3) void gemm_tile_kernel(FragMat w, const int8_t* __restrict__ aq,
                                                                    const uint16_t* __restrict__ ad, int m_rows,
                                                                    float* __restrict__ out, int ldo, int accumulate,
                                                                    int kbs, size_t split_stride, RowsEpi ep) {
    static_assert(EPI != RW_GATEUP || SN == 2, "the gate/up epilogue pairs two tiles");
    static_assert(D == 2 || D == 4, "two or four blocks of operands in flight");
    constexpr int NT = SM * SN;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int KB = w.k >> 5;
    const int fr = lane & 31, fh = lane >> 5;
    const int mtiles = (m_rows + 31) >> 5, ntiles = (w.rows + 31) >> 5, ffn = w.rows >> 1;
    const int mt0 = ((int)blockIdx.y * WM + wave / WN) * SM;
    const int nt0 = ((int)blockIdx.x * WN + wave % WN) * SN;
    const int gt = (int)blockIdx.x * WN + wave % WN;  // RW_GATEUP: the FFN block
    const int kb_begin = (int)blockIdx.z * kbs, kb_end = min(KB, kb_begin + kbs);
    out += blockIdx.z * split_stride;

    // Per tile: its first byte, bytes per block, this lane's offset in a block,
    // and the same for the scale words.  Tiles and rows past the end repeat the
    // last one; their results are not stored.
    const int8_t* pa[SM];
    const int8_t* pw[SN];
    const uint16_t* psa[SM];
    const uint16_t* psw[SN];
    int ra[SM], rw[SN];          // rows of the tile
    uint32_t va[SM], vw[SN];     // lane offsets, payload
    // this lane's row in a tile of rt rows (formed where it is used: held for
    // every tile it would take registers that the loop does not have)
    auto row_in = [&](int rt) {
        uint32_t r = fr;
        asm volatile("" : "+v"(r));
        return min(r, (uint32_t)(rt - 1));
    };
#pragma unroll
    for (int i = 0; i < SM; i++) {
        const int t = min(mt0 + i, mtiles - 1);
        ra[i] = frag_tile_rows(m_rows, 32 * t);
        pa[i] = aq + (size_t)t * 32 * w.k;
        psa[i] = ad + (size_t)t * 32 * KB;
        va[i] = (fh * ra[i] + row_in(ra[i])) * 16;
    }
#pragma unroll
    for (int j = 0; j < SN; j++) {
        const int t = EPI == RW_GATEUP ? j * (ffn >> 5) + min(gt, (ffn >> 5) - 1) : min(nt0 + j, ntiles - 1);
        rw[j] = frag_tile_rows(w.rows, 32 * t);
        pw[j] = w.q + (size_t)t * (WT == WT_Q8_0 ? 32 : 16) * w.k;
        psw[j] = w.s + (size_t)t * 32 * KB;
        vw[j] = ((WT == WT_Q8_0 ? fh * rw[j] : 0) + row_in(rw[j])) * 16;
    }
    struct Operands {
        sq_v4i a[SM], w[SN];
    };
    auto load = [&](Operands& S, int b) {
#pragma unroll
        for (int i = 0; i < SM; i++) S.a[i] = *(const sq_v4i*)lane_at(pa[i] + (size_t)b * (32 * ra[i]), va[i]);
#pragma unroll
        for (int j = 0; j < SN; j++)
            S.w[j] = *(const sq_v4i*)lane_at(pw[j] + (size_t)b * ((WT == WT_Q8_0 ? 32 : 16) * rw[j]), vw[j]);
    };
    // the scales of the block pair b, b + 1 (b even) of this lane's rows
    uint32_t sa[2][SM], sw[2][SN];
    auto load_scales = [&](int k, int b) {
#pragma unroll
        for (int i = 0; i < SM; i++) sa[k][i] = *(const uint32_t*)lane_at(psa[i] + (size_t)b * ra[i], 4 * row_in(ra[i]));
#pragma unroll
        for (int j = 0; j < SN; j++)
            sw[k][j] = *(const uint32_t*)lane_at(psw[j] + (size_t)b * rw[j], 4 * row_in(rw[j]));
    };
    m8_v16f acc[NT];
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[t][r] = 0.0f;
    const m8_v16i ibase = isum_base<m8_v16i>();
    const m8_v16f fzero = {};
    // k-slots 0 and 1 of lanes 0-31 carry the even and odd block's scale
    const uint32_t mask[2] = {fh ? 0u : 0x0000FFFFu, fh ? 0u : 0xFFFF0000u};
    const int sh = fh ? 0 : 4;  // Q4_0: this lane's nibbles
    auto compute = [&](const Operands& S, const uint32_t (&ssa)[SM], const uint32_t (&ssw)[SN], int h) {
        sq_v4i bw[SN];
#pragma unroll
        for (int j = 0; j < SN; j++) bw[j] = WT == WT_Q8_0 ? S.w[j] : q4_bytes(S.w[j], sh);
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const int i = t / SN, j = t % SN;
            const m8_v16i d = __builtin_amdgcn_mfma_i32_32x32x32_i8(S.a[i], bw[j], ibase, 0, 0, 0);
            const m8_v16f sc = __builtin_amdgcn_mfma_f32_32x32x8f16(
                __builtin_bit_cast(mq_v4h, make_uint2(ssa[i] & mask[h], 0u)),
                __builtin_bit_cast(mq_v4h, make_uint2(ssw[j] & mask[h], 0u)), fzero, 0, 0, 0);
            // the combine of the reference's aarch64 kernels (dot_prod.rs:189-252):
            // acc = fma(f32(isum), sa * sw, acc)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[t][r] = fmaf(isum_f32(d[r]), sc[r], acc[t][r]);
            // one tile's products live at a time (left to itself the scheduler
            // issues every product first and spills the results)
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // Groups of four blocks with the next blocks' loads in flight (clamped past
    // the matrix's end), then the blocks that remain, one at a time.
    const int b4 = kb_begin + ((kb_end - kb_begin) & ~3);
    if (b4 > kb_begin) {
        Operands S[D];
        const int last = KB - 1, last_pair = (KB & ~1) - 2;
        load_scales(0, kb_begin);
#pragma unroll
        for (int q = 0; q < D; q++) load(S[q], kb_begin + q);
        for (int b = kb_begin; b < b4; b += 4) {
#pragma unroll
            for (int u = 0; u < 4; u++) {
                if ((u & 1) == 0) load_scales(((u >> 1) + 1) & 1, min(b + u + 2, last_pair));
                __builtin_amdgcn_sched_barrier(0);
                compute(S[u % D], sa[u >> 1], sw[u >> 1], u & 1);
                load(S[u % D], min(b + u + D, last));
            }
        }
    }
    for (int b = b4; b < kb_end; b++) {
        Operands S;
        load(S, b);
        uint32_t xa[SM], xw[SN];
        // the scale's place among the pairs, or alone at an odd end
        const int odd = b & 1, solo = b == KB - 1 && !odd;
#pragma unroll
        for (int i = 0; i < SM; i++)
            xa[i] = psa[i][(size_t)(b & ~1) * ra[i] + (solo ? 1 : 2) * row_in(ra[i]) + odd];
#pragma unroll
        for (int j = 0; j < SN; j++)
            xw[j] = psw[j][(size_t)(b & ~1) * rw[j] + (solo ? 1 : 2) * row_in(rw[j]) + odd];
        compute(S, xa, xw, 0);
    }
    if constexpr (WT == WT_Q4_0) {
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[t][r] *= kOutScale<WT>;
    }

    if constexpr (EPI == RW_GATEUP) {
        // rows 36 floats apart: a lane's 16-byte reads of its row and the
        // 32 lanes' stores of a column run fall in distinct banks
        constexpr int LD = 36;
        __shared__ __attribute__((aligned(16))) float s_t[WM * WN][SM * 32][LD];
        float (*const tl)[LD] = s_t[wave];
#pragma unroll
        for (int i = 0; i < SM; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const float g = acc[SN * i][r], u = acc[SN * i + 1][r];
                tl[32 * i + 8 * (r >> 2) + 4 * fh + (r & 3)][fr] = (g * sq_sigmoid(g)) * u;  // (silu_mul8_kernel)
            }
        __syncthreads();
        if (SM == 1 && lane >= 32) return;
        const int m = 32 * mt0 + lane;
        if (m >= m_rows || gt >= (ffn >> 5)) return;
        float v[32];
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const sq_v4f x = *(const sq_v4f*)&tl[lane][4 * k];
            v[4 * k] = x.x;
            v[4 * k + 1] = x.y;
            v[4 * k + 2] = x.z;
            v[4 * k + 3] = x.w;
        }
        float mx = fabsf(v[0]);
#pragma unroll
        for (int k = 1; k < 32; k++) mx = fmaxf(mx, fabsf(v[k]));
        const float scale = sq_q8_scale(fmaxf(mx, 0.0f)), inv = sq_q8_inv(scale);
        unsigned q[8];
#pragma unroll
        for (int k = 0; k < 8; k++) {
            q[k] = 0;
#pragma unroll
            for (int c = 0; c < 4; c++) q[k] |= (unsigned)(uint8_t)sq_q8_quant(v[4 * k + c], inv) << (8 * c);
        }
        int8_t* const dst = ep.act_q + frag_q8(m_rows, ffn, m, gt);
        *(sq_v4i*)dst = sq_v4i{(int)q[0], (int)q[1], (int)q[2], (int)q[3]};
        *(sq_v4i*)(dst + 16 * frag_tile_rows(m_rows, m)) = sq_v4i{(int)q[4], (int)q[5], (int)q[6], (int)q[7]};
        ep.act_d[frag_scale(m_rows, ffn >> 5, m, gt)] = sq_f32_to_f16(scale);
        return;
    }
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int m = 32 * (mt0 + t / SN) + 8 * (r >> 2) + 4 * fh + (r & 3), n = 32 * (nt0 + t % SN) + fr;
            const float v = acc[t][r];
            if constexpr (EPI == RW_QKV) {
                const float pv = __shfl_xor(v, 1, 64);  // column n ^ 1 of the same prompt row
                if (m >= m_rows || n >= w.rows) continue;
                const int QD = ep.q_dim, KVD = ep.kv_dim, p = ep.pos0 + m;
                if (n < QD + KVD) {
                    const bool is_q = n < QD;
                    const int li = is_q ? n : n - QD;
                    const float2 cs = ep.rope[(size_t)p * (ep.head_dim >> 1) + ((li % ep.head_dim) >> 1)];
                    float o0, o1;
                    if (n & 1) sq_rotate(pv, v, cs.x, cs.y, o0, o1);
                    else sq_rotate(v, pv, cs.x, cs.y, o0, o1);
                    const float o = (n & 1) ? o1 : o0;
                    if (is_q) ep.q_out[(size_t)m * QD + li] = o;
                    else ep.kcache[(size_t)p * KVD + li] = o;
                } else {
                    ep.vcache[(size_t)p * KVD + (n - QD - KVD)] = v;
                }
            } else if (m < m_rows && n < w.rows) {
                float* o = out + (size_t)m * ldo + n;
                *o = accumulate ? *o + v : v;
            }
        }
}

// out[r, c] (+)= the sum of the K-split partial tiles, in split order.
__global__ __launch_bounds__(256) void split_sum_kernel(const float* __restrict__ ws, int splits, size_t stride,
                                                        int m, int n, float* __restrict__ out, int ldo,
                                                        int accumulate) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (size_t)m * n) return;
    float v = 0.0f;
    for (int z = 0; z < splits; z++) v += ws[z * stride + i];
    float* o = out + (i / n) * (size_t)ldo + i % n;
    *o = accumulate ? *o + v : v;
}

// The same sums four elements per thread (16-byte loads and stores) where
// n, ldo and stride are multiples of 4 and the buffers 16-byte aligned.
__global__ __launch_bounds__(256) void split_sum4_kernel(const float* __restrict__ ws, int splits, size_t stride,
                                                         int m, int n, float* __restrict__ out, int ldo,
                                                         int accumulate) {
    const size_t i = 4 * ((size_t)blockIdx.x * 256 + threadIdx.x);
    if (i >= (size_t)m * n) return;
    float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    for (int z = 0; z < splits; z++) {
        const float4 p = *(const float4*)(ws + z * stride + i);
        v.x += p.x;
        v.y += p.y;
        v.z += p.z;
        v.w += p.w;
    }
    float4* o = (float4*)(out + (i / n) * (size_t)ldo + i % n);
    if (accumulate) {
        const float4 a = *o;
        v = make_float4(a.x + v.x, a.y + v.y, a.z + v.z, a.w + v.w);
    }
    *o = v;
}

// The stacked q|k|v projection's K-split partials ([m][ncols] each, stride
// apart) summed in split order as split_sum_kernel sums them, then RoPE on the
// q and k columns and the KV-cache append as rope_kv_kernel applies them: a
// workgroup takes 1024 columns of a prompt row, a thread two RoPE pairs (one
// workgroup a row with a pair per thread and load took 9.3 us for 301 rows).
// q_dim, kv_dim and head_dim are multiples of 4; the buffers 16-byte aligned.
__global__ __launch_bounds__(256) void split_sum_rope_kernel(const float* __restrict__ ws, int splits, size_t stride,
                                                             int ncols, RowsEpi ep) {
    const int m = blockIdx.x, p = ep.pos0 + m;
    const int e = 4 * (256 * (int)blockIdx.y + (int)threadIdx.x);
    if (e >= ncols) return;
    const int QD = ep.q_dim, KVD = ep.kv_dim, half = ep.head_dim >> 1;
    const bool is_q = e < QD, is_v = e >= QD + KVD;
    const int li = is_q ? e : is_v ? e - QD - KVD : e - QD;
    const float4 cs = is_v ? make_float4(0.f, 0.f, 0.f, 0.f)
                           : *(const float4*)(ep.rope + (size_t)p * half + ((li % ep.head_dim) >> 1));
    const float* src = ws + (size_t)m * ncols + e;
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int z = 0; z < splits; z++) {
        const float4 x = *(const float4*)(src + z * stride);
        v.x += x.x;
        v.y += x.y;
        v.z += x.z;
        v.w += x.w;
    }
    if (is_v) {
        *(float4*)(ep.vcache + (size_t)p * KVD + li) = v;
        return;
    }
    float4 o;
    sq_rotate(v.x, v.y, cs.x, cs.y, o.x, o.y);
    sq_rotate(v.z, v.w, cs.z, cs.w, o.z, o.w);
    *(float4*)(is_q ? ep.q_out + (size_t)m * QD + li : ep.kcache + (size_t)p * KVD + li) = o;
}

// out (+)= the split partials in split order, on the vector kernel where the
// shapes and buffers allow it.
// With *then, the norm of the rows that follows goes into the same launch where
// that kernel takes them (and *then becomes null: done).
int launch_split_sum(hipStream_t s, const float* ws, int splits, size_t stride, int m, int n, float* out, int ldo,
                     bool acc, const NormThen** then) {
    if (*then && acc && ldo == n && norm8_fits(n) && stride % 4 == 0 &&
        (((uintptr_t)ws | (uintptr_t)out | (uintptr_t)(*then)->w) & 15) == 0) {
        const int st = launch_split_sum_norm(s, ws, splits, stride, m, n, out, **then);
        *then = nullptr;
        return st;
    }
    const size_t total = (size_t)m * n;
    if (n % 4 == 0 && ldo % 4 == 0 && stride % 4 == 0 && (((uintptr_t)ws | (uintptr_t)out) & 15) == 0)
        hipLaunchKernelGGL(split_sum4_kernel, dim3((unsigned)((total / 4 + 255) / 256)), dim3(256), 0, s, ws, splits,
                           stride, m, n, out, ldo, acc ? 1 : 0);
    else
        hipLaunchKernelGGL(split_sum_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, ws, splits,
                           stride, m, n, out, ldo, acc ? 1 : 0);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return set_error(SQ_ERR_HIP, std::string("split sum launch: ") + hipGetErrorString(e));
    return 0;
}

// ---- few activation rows: the weights streamed once --------------------------
// A prompt of a few dozen rows (the short prompts of a generation) makes the
// matmul a weight stream with little arithmetic per byte.  Here a
// workgroup takes 32 activation rows and NT tiles of 32 weight rows: one
// v_mfma_i32_32x32x32_i8 per block and tile (lane l supplies 16 bytes of row
// l % 32, half l / 32 of the block; activations as operand A, weights as
// operand B) and one v_mfma_f32_32x32x8f16 for the scale products sa * sw
// (lanes 0-31 hold the row's and the column's scale in k-slot 0, the others
// zeros).  Its RW_NW wavefronts take consecutive ranges of the workgroup's
// K, each with two batches of RW_NB blocks of loads in flight (branch-free:
// blocks past a range read a clamped address and get zero scales), and sum
// their partial tiles through LDS in wavefront order.  A long K on a narrow
// matrix is also split over workgroups (blockIdx.z), whose partial tiles
// split_sum_kernel adds in split order.  The per-block combine is that of
// the other kernels: fma(f32(isum), sa * sw, acc) (dot_prod.rs:189-252).
//
// Epilogues (EPI): RW_STORE writes (or adds) the tile.  RW_GATEUP: the FFN
// gate/up projection with SiLU(gate) * up and its Q8_0 blocks (two tiles:
// gate rows 32 j.. and the up rows ffn + 32 j..); a 32-lane half of a
// wavefront then holds one prompt row's 32 values of FFN block j and forms
// the block as silu_mul8_kernel does.  RW_QKV: the stacked q|k|v projection
// with RoPE on q and k and the KV-cache append, as rope_kv_kernel does (the
// pair partner of column n is column n ^ 1, lane l ^ 1).  The same
// operations on the same values, so the same bits as the separate kernels.
constexpr int RW_NW = 8;  // wavefronts per workgroup
constexpr int RW_NB = 4;  // blocks per load batch

template <int NT, int NB>
struct RwBatch {
    sq_v4i w[NT][NB];  // Q8_0: 16 bytes of the block; Q4_0: the packed block
    sq_v4i a[NB];
    uint32_t sw[NT][NB / 2], sa[NB / 2];  // f16 scales of block pairs: this lane's weight rows, its activation row
};

template <int WT, int NT, int NB, int EPI>
__global__ __launch_bounds__(RW_NW * 64) void gemm_rows_kernel(FragMat w, const int8_t* __restrict__ aq,
                                                               const uint16_t* __restrict__ ad, int m_rows,
                                                               float* __restrict__ out, int ldo, int accumulate,
                                                               int per, int kbs, size_t split_stride, RowsEpi ep,
                                                               SharedMats more) {
    constexpr bool GU = EPI == RW_GATEUP;
    int bx = blockIdx.x;
    if constexpr (EPI == RW_SHARED) {
#pragma unroll
        for (int i = kSharedMax - 2; i >= 0; i--)
            if (bx >= more.begin[i]) {
                w = more.w[i];
                out = more.out[i];
                ldo = w.rows;
                bx -= more.begin[i];
                break;
            }
    }
    static_assert(!GU || NT == 2, "the gate/up epilogue pairs two tiles");
    static_assert(EPI != RW_QKV || NT == 1, "the q|k|v epilogue takes one tile");
    __shared__ float red[RW_NW][NT * 16][64];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int K = w.k, KB = K >> 5;
    const int n0 = bx * 32 * NT, m0 = blockIdx.y * 32;
    const int fr = lane & 31, fh = lane >> 5;
    // the workgroup's blocks [kb_begin, kb_end) (split blockIdx.z), and this
    // wavefront's [kbw, kend): per (a multiple of 2 NB) per wavefront
    const int kb_begin = blockIdx.z * kbs, kb_end = min(KB, kb_begin + kbs);
    out += blockIdx.z * split_stride;
    const int kbw = kb_begin + wave * per, kend = min(kb_end, kbw + per);
    const int nb = per / NB;
    typedef RwBatch<NT, NB> Batch;
    // Operands in fragment order (sq_common.h): per tile its first byte, its
    // rows and this lane's offsets.  Rows and tiles past the end repeat the last
    // one; their results are not stored.
    const int ffn = w.rows / 2, j0 = bx * 32;  // GU: the FFN block's first column
    const int8_t* pw[NT];
    const uint16_t* psw[NT];
    int rw[NT];
    uint32_t vw[NT], uw[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) {
        const int tile = GU ? t * (ffn >> 5) + bx : min(NT * bx + t, (w.rows - 1) >> 5);
        rw[t] = frag_tile_rows(w.rows, 32 * tile);
        pw[t] = w.q + (size_t)tile * (WT == WT_Q8_0 ? 32 : 16) * K;
        psw[t] = w.s + (size_t)tile * 32 * KB;
        uw[t] = min(fr, rw[t] - 1);
        vw[t] = (WT == WT_Q8_0 ? fh * rw[t] + uw[t] : uw[t]) * 16;
    }
    const int ra = frag_tile_rows(m_rows, m0);
    const int8_t* const pa = aq + (size_t)m0 * K;
    const uint16_t* const psa = ad + (size_t)m0 * KB;
    const uint32_t ua = min(fr, ra - 1), va = (fh * ra + ua) * 16;
    const int sh = fh ? 0 : 4;  // Q4_0: this lane's nibbles

    auto load = [&](Batch& B, int kb) {
        const int kc = min(kb, KB - NB);  // KB is a multiple of NB
#pragma unroll
        for (int j = 0; j < NB; j++) {
#pragma unroll
            for (int t = 0; t < NT; t++)
                B.w[t][j] =
                    *(const sq_v4i*)lane_at(pw[t] + (size_t)(kc + j) * ((WT == WT_Q8_0 ? 32 : 16) * rw[t]), vw[t]);
            B.a[j] = *(const sq_v4i*)lane_at(pa + (size_t)(kc + j) * (32 * ra), va);
        }
#pragma unroll
        for (int j = 0; j < NB; j += 2) {
#pragma unroll
            for (int t = 0; t < NT; t++)
                B.sw[t][j / 2] = *(const uint32_t*)lane_at(psw[t] + (size_t)(kc + j) * rw[t], 4 * uw[t]);
            B.sa[j / 2] = *(const uint32_t*)lane_at(psa + (size_t)(kc + j) * ra, 4 * ua);
        }
    };
    m8_v16f acc[NT];
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[t][r] = 0.0f;
    const m8_v16i ibase = isum_base<m8_v16i>();
    const m8_v16f fzero = {};
    auto compute = [&](const Batch& B, int kb) {
#pragma unroll
        for (int j = 0; j < NB; j++) {
            // blocks past the range fold nothing: both scales zero (an
            // activation scale may be inf, and inf * 0 would not be).
            // (masks, not branches: a branch here lets the compiler move
            // every block's combine after all the matrix instructions)
            const uint32_t mask = kb + j < kend && fh == 0 ? ((j & 1) ? 0xFFFF0000u : 0x0000FFFFu) : 0u;
            const mq_v4h sa = __builtin_bit_cast(mq_v4h, make_uint2(B.sa[j / 2] & mask, 0u));
#pragma unroll
            for (int t = 0; t < NT; t++) {
                const sq_v4i wf = WT == WT_Q8_0 ? B.w[t][j] : q4_bytes(B.w[t][j], sh);
                const mq_v4h sw = __builtin_bit_cast(mq_v4h, make_uint2(B.sw[t][j / 2] & mask, 0u));
                const m8_v16i d = __builtin_amdgcn_mfma_i32_32x32x32_i8(B.a[j], wf, ibase, 0, 0, 0);
                const m8_v16f sc = __builtin_amdgcn_mfma_f32_32x32x8f16(sa, sw, fzero, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 16; r++) acc[t][r] = fmaf(isum_f32(d[r]), sc[r], acc[t][r]);
                // one tile's products live at a time: left to itself the
                // scheduler issues every block's matrix instructions first and
                // spills their results
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };
    Batch B0, B1;
    load(B0, kbw);
    load(B1, kbw + NB);
    for (int b = 0; b + 2 < nb; b += 2) {
        compute(B0, kbw + b * NB);
        load(B0, kbw + (b + 2) * NB);
        compute(B1, kbw + (b + 1) * NB);
        load(B1, kbw + (b + 3) * NB);
    }
    compute(B0, kbw + (nb - 2) * NB);
    compute(B1, kbw + (nb - 1) * NB);

    // partial tiles summed in wavefront order; element r of lane l of tile t
    // is row 8 (r / 4) + 4 (l / 32) + r % 4, column 32 t + l % 32
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int r = 0; r < 16; r++) red[wave][16 * t + r][lane] = acc[t][r] * kOutScale<WT>;
    __syncthreads();
    if constexpr (GU) {
        // e = 64 r + l: lanes l < 32 and l >= 32 of a wavefront are two
        // prompt rows' FFN block j (column l % 32)
        for (int e = tid; e < 16 * 64; e += RW_NW * 64) {
            const int r = e >> 6, l = e & 63;
            float g = 0.0f, u = 0.0f;
#pragma unroll
            for (int q = 0; q < RW_NW; q++) {
                g += red[q][r][l];
                u += red[q][16 + r][l];
            }
            const float v = (g * sq_sigmoid(g)) * u;  // silu(gate) * up (silu_mul8_kernel)
            float mx = fabsf(v);
#pragma unroll
            for (int o = 16; o >= 1; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
            const float scale = sq_q8_scale(fmaxf(mx, 0.0f)), inv = sq_q8_inv(scale);
            const int mm = m0 + 8 * (r >> 2) + 4 * (l >> 5) + (r & 3), jj = l & 31;
            if (mm < m_rows && j0 + jj < ffn) {
                ep.act_q[frag_q8(m_rows, ffn, mm, bx) + (size_t)(jj >> 4) * 16 * frag_tile_rows(m_rows, mm) +
                         (jj & 15)] = sq_q8_quant(v, inv);
                if (jj == 0) ep.act_d[frag_scale(m_rows, ffn / 32, mm, bx)] = sq_f32_to_f16(scale);
            }
        }
        return;
    }
    if constexpr (EPI == RW_QKV) {
        for (int e = tid; e < 16 * 64; e += RW_NW * 64) {
            const int r = e >> 6, l = e & 63;
            float v = 0.0f;
#pragma unroll
            for (int q = 0; q < RW_NW; q++) v += red[q][r][l];
            const float pv = __shfl_xor(v, 1, 64);  // column n ^ 1 of the same prompt row
            const int mm = m0 + 8 * (r >> 2) + 4 * (l >> 5) + (r & 3), n = n0 + (l & 31);
            if (mm >= m_rows || n >= w.rows) continue;
            const int QD = ep.q_dim, KVD = ep.kv_dim, p = ep.pos0 + mm;
            if (n < QD + KVD) {
                const bool is_q = n < QD;
                const int li = is_q ? n : n - QD;
                const float2 cs = ep.rope[(size_t)p * (ep.head_dim >> 1) + ((li % ep.head_dim) >> 1)];
                float o0, o1;
                if (n & 1) sq_rotate(pv, v, cs.x, cs.y, o0, o1);
                else sq_rotate(v, pv, cs.x, cs.y, o0, o1);
                const float o = (n & 1) ? o1 : o0;
                if (is_q) ep.q_out[(size_t)mm * QD + li] = o;
                else ep.kcache[(size_t)p * KVD + li] = o;
            } else {
                ep.vcache[(size_t)p * KVD + (n - QD - KVD)] = v;
            }
        }
        return;
    }
    for (int e = tid; e < NT * 16 * 64; e += RW_NW * 64) {
        const int tr = e >> 6, l = e & 63, t = tr >> 4, r = tr & 15;
        float v = 0.0f;
#pragma unroll
        for (int q = 0; q < RW_NW; q++) v += red[q][tr][l];
        const int mm = m0 + 8 * (r >> 2) + 4 * (l >> 5) + (r & 3), nn = n0 + 32 * t + (l & 31);
        if (mm < m_rows && nn < w.rows) {
            float* o = out + (size_t)mm * ldo + nn;
            *o = accumulate ? *o + v : v;
        }
    }
}

// Compute units of the current device (the grid-size rules below are in
// workgroups per CU).
int device_cus() {
    static int cus[64] = {};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    if (cus[dev] == 0) {
        int n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
        cus[dev] = n;
    }
    return cus[dev];
}

// The tile shapes: 128 x 128 outputs a workgroup (four wavefronts of 64 x 64),
// 128 x 64 (four of 32 x 64), 64 x 64 (two of 32 x 64) and 64 x 128 (four).
// All fold the same per-block terms in the same order.
enum : int { SHAPE_128, SHAPE_128X64, SHAPE_64, SHAPE_64X128, SHAPE_ROWS };  // (the last: the few-rows kernel)
int shape_rows(int shape) { return shape == SHAPE_128 || shape == SHAPE_128X64 ? 128 : 64; }
int shape_cols(int shape) { return shape == SHAPE_128 || shape == SHAPE_64X128 ? 128 : 64; }

// Matmul launches since the last reset (measurement aid): all, K-split, the
// largest split count, and by shape.
std::atomic<uint64_t> g_launches{0}, g_split_launches{0}, g_max_splits{0}, g_shape_launches[SHAPE_ROWS + 1]{};
void count_launch(int splits, int shape) {
    g_launches++;
    g_shape_launches[shape]++;
    if (splits > 1) g_split_launches++;
    uint64_t prev = g_max_splits.load();
    while ((uint64_t)splits > prev && !g_max_splits.compare_exchange_weak(prev, (uint64_t)splits)) {
    }
}

FragMat frag(const DevMatrix& w) { return FragMat{(const int8_t*)w.fq, w.fs, w.rows, w.k}; }

template <int WT, int EPI>
int launch_shape(hipStream_t s, int shape, const DevMatrix& w, const int8_t* aq, const uint16_t* ad, int m, float* out,
                 int ldo, bool acc, int splits, int kbs, size_t stride, const RowsEpi& ep = RowsEpi{}) {
    const dim3 grid((w.rows + shape_cols(shape) - 1) / shape_cols(shape), (m + shape_rows(shape) - 1) / shape_rows(shape),
                    splits);
#define SQ_TILE_LAUNCH(SM, SN, WM, WN, D)                                                                          \
    hipLaunchKernelGGL((gemm_tile_kernel<WT, SM, SN, WM, WN, D, EPI>), grid, dim3(64 * WM * WN), 0, s, frag(w), aq, \
                       ad, m, out, ldo, acc ? 1 : 0, kbs, stride, ep)
    switch (shape) {
        case SHAPE_128: SQ_TILE_LAUNCH(2, 2, 2, 2, 2); break;
        case SHAPE_128X64: SQ_TILE_LAUNCH(1, 2, 4, 1, 2); break;
        case SHAPE_64X128: SQ_TILE_LAUNCH(1, 2, 2, 2, 2); break;
        default:
            if constexpr (EPI == RW_GATEUP) SQ_TILE_LAUNCH(1, 2, 2, 1, 4);
            else SQ_TILE_LAUNCH(1, 1, 2, 2, 4);
            break;
    }
#undef SQ_TILE_LAUNCH
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return set_error(SQ_ERR_HIP, std::string("gemm launch: ") + hipGetErrorString(e));
    return 0;
}

// Blocks per split and the splits that leaves, for `splits` splits of K in
// whole groups of four blocks (the loop's; three splits of 64 blocks are 24, 24
// and 16).  The parts fix the order of the sums and so a product's last bits.
void k_partition(int KB, int* splits, int* kbs) {
    const int groups = (KB + 3) / 4;
    *kbs = ((groups + *splits - 1) / *splits) * 4;
    *splits = (KB + *kbs - 1) / *kbs;
}

// A product on one tile shape with K split `splits` ways (the partials in ws,
// summed in split order, so results do not depend on scheduling).
template <int WT>
int run_tiles(hipStream_t s, int shape, const DevMatrix& w, const int8_t* aq, const uint16_t* ad, int m, float* out,
              int ldo, bool acc, int splits, float* ws, const NormThen** then) {
    int kbs;
    k_partition(w.k / 32, &splits, &kbs);
    count_launch(splits, shape);
    if (splits == 1) return launch_shape<WT, RW_STORE>(s, shape, w, aq, ad, m, out, ldo, acc, 1, kbs, 0);
    const size_t stride = (size_t)m * w.rows;
    if (const int st = launch_shape<WT, RW_STORE>(s, shape, w, aq, ad, m, ws, w.rows, false, splits, kbs, stride)) return st;
    return launch_split_sum(s, ws, splits, stride, m, w.rows, out, ldo, acc, then);
}

// Splits for a grid of `tiles` workgroups on which `target` are wanted, within
// the workspace.
int splits_for(const DevMatrix& w, int m, int tiles, int target, float* ws, size_t ws_floats) {
    if (ws == nullptr || tiles >= target) return 1;
    int splits = min((w.k / 32 + 3) / 4, (target + tiles - 1) / tiles);
    while (splits > 1 && (size_t)splits * m * w.rows > ws_floats) splits--;
    return splits;
}

// K per wavefront of the few-rows kernel, kbs blocks in all.
int rows_per_wave(int kbs, int NB) { return ((kbs + RW_NW - 1) / RW_NW + 2 * NB - 1) / (2 * NB) * (2 * NB); }
// The few-rows kernel: grid (column tiles of 32 NT, row tiles of 32, K
// splits), K in blocks of 32 with KB a multiple of RW_NB.  Two column tiles
// per workgroup where that still gives every CU a workgroup (the FFN gate/up
// projection: twice the weights in flight per CU, one round of the grid); a
// K split where the grid has fewer workgroups than CUs and each split keeps
// two full batches per wavefront (the FFN down projection, K = 8192: four
// splits).
template <int WT, int NT, int EPI = RW_STORE>
int launch_rows(hipStream_t s, const DevMatrix& w, const int8_t* aq, const uint16_t* ad, int m, float* out, int ldo,
                bool acc, int gx, int gy, int splits, int kbs, float* ws, const RowsEpi& ep = RowsEpi{},
                const NormThen** then = nullptr) {
    constexpr int NB = RW_NB;
    const int per = rows_per_wave(kbs, NB);
    if (splits == 1) {
        hipLaunchKernelGGL((gemm_rows_kernel<WT, NT, NB, EPI>), dim3(gx, gy), dim3(RW_NW * 64), 0, s, frag(w), aq, ad, m, out,
                           ldo, acc ? 1 : 0, per, kbs, (size_t)0, ep, SharedMats{});
    } else {
        const size_t stride = (size_t)m * w.rows;
        hipLaunchKernelGGL((gemm_rows_kernel<WT, NT, NB, RW_STORE>), dim3(gx, gy, splits), dim3(RW_NW * 64), 0, s, frag(w), aq,
                           ad, m, ws, w.rows, 0, per, kbs, stride, RowsEpi{}, SharedMats{});
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return set_error(SQ_ERR_HIP, std::string("gemm launch: ") + hipGetErrorString(e));
        if (const int st = launch_split_sum(s, ws, splits, stride, m, w.rows, out, ldo, acc, then)) return st;
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return set_error(SQ_ERR_HIP, std::string("gemm launch: ") + hipGetErrorString(e));
    return 0;
}

struct RowsPlan {
    bool two;  // two column tiles per workgroup
    int gx, gy, splits;
};
RowsPlan rows_plan(const DevMatrix& w, int m, bool have_ws, size_t ws_floats) {
    const int KB = w.k / 32, cus = device_cus();
    const int gy = (m + 31) / 32, tiles = (w.rows + 31) / 32;
    RowsPlan p{(tiles + 1) / 2 * gy >= cus, 0, gy, 1};
    p.gx = p.two ? (tiles + 1) / 2 : tiles;
    if (have_ws && p.gx * gy < cus) {
        int splits = min((cus + p.gx * gy - 1) / (p.gx * gy), KB / (RW_NW * 2 * RW_NB));
        while (splits > 1 && ((size_t)splits * m * w.rows > ws_floats || KB % splits || (KB / splits) % RW_NB))
            splits--;
        p.splits = max(splits, 1);
    }
    return p;
}

template <int WT>
int run_rows_shared(hipStream_t s, const DevMatrix* const* ws, int n, const int8_t* aq, const uint16_t* ad, int m,
                    float* const* outs) {
    SharedMats more{};
    int gx = 0;
    for (int i = 0; i < n; i++) {
        if (i > 0) {
            more.w[i - 1] = frag(*ws[i]);
            more.out[i - 1] = outs[i];
            more.begin[i - 1] = gx;
        }
        gx += (ws[i]->rows + 31) / 32;
        count_launch(1, SHAPE_ROWS);
    }
    for (int i = n - 1; i < kSharedMax - 1; i++) more.begin[i] = gx;  // (past the grid)
    const int KB = ws[0]->k / 32;
    hipLaunchKernelGGL((gemm_rows_kernel<WT, 1, RW_NB, RW_SHARED>), dim3(gx, (m + 31) / 32), dim3(RW_NW * 64), 0, s,
                       frag(*ws[0]), aq, ad, m, outs[0], ws[0]->rows, 0, rows_per_wave(KB, RW_NB), KB, (size_t)0,
                       RowsEpi{}, more);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return set_error(SQ_ERR_HIP, std::string("gemm launch: ") + hipGetErrorString(e));
    return 0;
}

template <int WT>
int run_rows(hipStream_t s, const DevMatrix& w, const int8_t* aq, const uint16_t* ad, int m, float* out, int ldo,
             bool acc, float* ws, size_t ws_floats, const NormThen** then) {
    const RowsPlan p = rows_plan(w, m, ws != nullptr, ws_floats);
    const bool two = p.two;
    const int KB = w.k / 32, gx = p.gx, gy = p.gy, splits = p.splits;
    const int kbs = KB / splits;
    count_launch(splits, SHAPE_ROWS);
    return two ? launch_rows<WT, 2>(s, w, aq, ad, m, out, ldo, acc, gx, gy, splits, kbs, ws, RowsEpi{}, then)
               : launch_rows<WT, 1>(s, w, aq, ad, m, out, ldo, acc, gx, gy, splits, kbs, ws, RowsEpi{}, then);
}

// SQUIRREL_GEMM_TILE pins the prefill matmul's kernel (a test and
// measurement aid): "64", "64x128", "128x64" and "128" the tile kernel on 64 x 64,
// 64 x 128, 128 x 64 or 128 x 128 tiles, "rows" the few-rows kernel.  Unset, inputs of at
// most 32 rows take the few-rows kernel, and larger ones auto_tiling's shape.
enum : int { TILE_AUTO, TILE_64, TILE_64X128, TILE_128X64, TILE_128, TILE_ROWS };
int gemm_tile_override() {
    const char* e = getenv("SQUIRREL_GEMM_TILE");
    if (!e) return TILE_AUTO;
    if (!strcmp(e, "64")) return TILE_64;
    if (!strcmp(e, "64x128")) return TILE_64X128;
    if (!strcmp(e, "128x64")) return TILE_128X64;
    if (!strcmp(e, "128")) return TILE_128;
    if (!strcmp(e, "rows")) return TILE_ROWS;
    return TILE_AUTO;
}

// Inputs the few-rows kernel takes unless a tiling is pinned: up to 32 rows.
bool rows_kernel_fits(int m, int k) { return m <= 32 && (k / 32) % RW_NB == 0 && gemm_tile_override() == TILE_AUTO; }

// The tile shape and K splits of an input past the few-rows kernel with no
// tiling pinned, shared by the plain path and the fused epilogues so that both
// fold the same terms:
//  - matrices of 8192 and more rows whose input would leave an eighth of its
//    128-row tiles empty: 64-row tiles, unsplit, from one and a half workgroups
//    per CU on (a wavefront of 32 x 64 spends 14% more per output than one of
//    64 x 64: 156 against 137 us for 2048 x 16384 x 2048; of 320 rows, 384 in
//    128-row tiles, 37 against 41);
//  - 128 x 128 tiles where they give every CU two workgroups;
//  - where they give one to two (on 256 CUs 256 to 511 tiles, a third to two
//    thirds of the three-per-CU slots) and the matrix has fewer than 8192 rows,
//    the same tiles with K split two or three ways, the partials summed in
//    split order: the o and FFN down projections of a 2048-token prompt (256
//    tiles) three ways, its q|k|v projection (384 tiles) two, every slot
//    taken once.  Counts that do not divide the slots leave the last ones empty
//    (q|k|v of 1800 rows, 360 tiles in three splits: 51 us alone, 46 in two);
//  (8192 rows stand between the 1B model's gate/up projection, 16384, and its
//  others, at most 3072; nothing lies between in a model.  On 8160 rows, which
//  the rule splits, 700 input rows take 47 us and 35 on unsplit 64 x 128 tiles:
//  the line is not drawn where the two meet)
//  - 128 x 64 tiles where those give every CU two workgroups;
//  - else 64 x 64 tiles, and where these are fewer than the CUs, K split over
//    about two workgroups per CU.
struct Tiling {
    int shape, splits;
};
Tiling auto_tiling(const DevMatrix& w, int m, float* ws, size_t ws_floats) {
    const int cus = device_cus(), gy = (m + 127) / 128, gy64 = (m + 63) / 64;
    const int g = (w.rows + 127) / 128 * gy, g64 = (w.rows + 63) / 64 * gy64;
    if (w.rows >= 8192 && 128 * gy * 7 >= 64 * gy64 * 8 && 2 * ((w.rows + 127) / 128 * gy64) >= 3 * cus)
        return {SHAPE_64X128, 1};
    if (m >= 128) {
        if (g >= 2 * cus) return {SHAPE_128, 1};
        if (w.k / 32 >= 64 && ws != nullptr && w.rows < 8192) {
            const int splits = (3 * cus + g - 1) / g;
            if (splits <= 3 && (size_t)splits * m * w.rows <= ws_floats) return {SHAPE_128, splits};
        }
        if ((w.rows + 63) / 64 * gy >= 2 * cus) return {SHAPE_128X64, 1};
    }
    return {SHAPE_64, g64 < cus ? splits_for(w, m, g64, 2 * cus, ws, ws_floats) : 1};
}

template <int WT>
int run_integer(hipStream_t s, const DevMatrix& w, const int8_t* aq, const uint16_t* ad, int m, float* out, int ldo,
                bool acc, float* ws, size_t ws_floats, const NormThen** then) {
    const int tile = gemm_tile_override();
    if ((tile == TILE_ROWS && (w.k / 32) % RW_NB == 0) || rows_kernel_fits(m, w.k))
        return run_rows<WT>(s, w, aq, ad, m, out, ldo, acc, ws, ws_floats, then);
    Tiling t = auto_tiling(w, m, ws, ws_floats);
    if (tile != TILE_AUTO && tile != TILE_ROWS) {
        // pinned: K split below two (64 x 64 tiles: one) workgroups per CU
        const int cus = device_cus(), shape = tile == TILE_128     ? SHAPE_128
                                              : tile == TILE_128X64 ? SHAPE_128X64
                                              : tile == TILE_64X128 ? SHAPE_64X128
                                                                    : SHAPE_64;
        const int g = (w.rows + shape_cols(shape) - 1) / shape_cols(shape) *
                      ((m + shape_rows(shape) - 1) / shape_rows(shape));
        t = Tiling{shape, shape == SHAPE_64 && g >= cus ? 1 : splits_for(w, m, g, 2 * cus, ws, ws_floats)};
    }
    return run_tiles<WT>(s, t.shape, w, aq, ad, m, out, ldo, acc, t.splits, ws, then);
}

// A matrix without a fragment-order copy (there was no room for it): the copy
// of as many rows as the workspace holds at a time, each slab's product unsplit.
template <int WT>
int run_slabs(hipStream_t s, const DevMatrix& w, const int8_t* aq, const uint16_t* ad, int m, float* out, int ldo,
              bool acc, float* ws, size_t ws_floats) {
    const size_t KB = w.k / 32, pay = KB * (WT == WT_Q8_0 ? 32 : 16), room = ws ? ws_floats * sizeof(float) : 0;
    size_t slab = room > 256 ? (room - 256) / (pay + 2 * KB) : 0;  // (256: the scales' boundary)
    if (slab >= 32) slab &= ~(size_t)31;
    if (slab == 0) return set_error(SQ_ERR_HIP, "gemm: the matrix has no fragment-order copy and the workspace no room for a row");
    for (size_t n0 = 0; n0 < (size_t)w.rows; n0 += slab) {
        DevMatrix part = w;
        part.rows = (int)min(slab, (size_t)w.rows - n0);
        part.qs = (uint8_t*)w.qs + n0 * pay;
        part.scale = w.scale + n0 * KB;
        part.fq = ws;
        part.fs = (uint16_t*)((uint8_t*)ws + (part.rows * pay + 255) / 256 * 256);
        if (const int st = launch_frag_copy(s, part)) return st;
        const NormThen* none = nullptr;
        if (const int st = run_integer<WT>(s, part, aq, ad, m, out + n0, ldo, acc, nullptr, 0, &none)) return st;
    }
    return 0;
}

// SQUIRREL_PREFILL_UNFUSED=1 turns the fused gate/up and q|k|v epilogues
// off (a test aid: the separate kernels give the same bits).
bool prefill_fusion_enabled() {
    const char* e = getenv("SQUIRREL_PREFILL_UNFUSED");
    return !(e && !strcmp(e, "1"));
}

// The FFN gate/up projection with SiLU * up and its Q8_0 blocks fused (one
// launch instead of two), on the kernel and tiles the plain path would take
// without a K split; -1 when it does not apply.
template <int WT>
int run_gateup_silu(hipStream_t s, const DevMatrix& w, const int8_t* aq, const uint16_t* ad, int m, int8_t* act_q,
                    uint16_t* act_d, float* ws, size_t ws_floats) {
    const int ffn = w.rows / 2, KB = w.k / 32;
    if (w.rows % 2 || ffn % 32 || !prefill_fusion_enabled()) return -1;
    RowsEpi ep{};
    ep.act_q = act_q;
    ep.act_d = act_d;
    if (!rows_kernel_fits(m, w.k)) {
        if (gemm_tile_override() != TILE_AUTO) return -1;
        const Tiling t = auto_tiling(w, m, ws, ws_floats);
        if (t.splits != 1) return -1;
        count_launch(1, t.shape);
        return launch_shape<WT, RW_GATEUP>(s, t.shape, w, aq, ad, m, nullptr, 0, false, 1, (KB + 1) & ~1, 0, ep);
    }
    const int gx = ffn / 32, gy = (m + 31) / 32;
    if (gx * gy < device_cus()) return -1;  // the split-free two-tile form only
    count_launch(1, SHAPE_ROWS);
    return launch_rows<WT, 2, RW_GATEUP>(s, w, aq, ad, m, nullptr, 0, false, gx, gy, 1, KB, nullptr, ep);
}

// The stacked q|k|v projection with RoPE and the KV-cache append fused: in the
// matmul's epilogue, or in the launch that sums its K-split partials; -1 when
// it does not apply.
template <int WT>
int run_qkv_rope(hipStream_t s, const DevMatrix& w, const int8_t* aq, const uint16_t* ad, int m, const RowsEpi& ep,
                 float* ws, size_t ws_floats) {
    const int KB = w.k / 32, gx = (w.rows + 31) / 32, gy = (m + 31) / 32;
    if (ep.head_dim % 2 || (ep.q_dim + ep.kv_dim) % 2 || w.rows != ep.q_dim + 2 * ep.kv_dim ||
        !prefill_fusion_enabled())
        return -1;
    if (!rows_kernel_fits(m, w.k)) {
        if (gemm_tile_override() != TILE_AUTO) return -1;
        Tiling t = auto_tiling(w, m, ws, ws_floats);
        int kbs;
        k_partition(KB, &t.splits, &kbs);
        // (four columns per thread of the summing kernel)
        if (t.splits > 1 && (ep.q_dim % 4 || ep.kv_dim % 4 || ep.head_dim % 4)) return -1;
        count_launch(t.splits, t.shape);
        if (t.splits == 1)
            return launch_shape<WT, RW_QKV>(s, t.shape, w, aq, ad, m, nullptr, 0, false, 1, kbs, 0, ep);
        const size_t stride = (size_t)m * w.rows;
        if (const int st = launch_shape<WT, RW_STORE>(s, t.shape, w, aq, ad, m, ws, w.rows, false, t.splits, kbs, stride))
            return st;
        hipLaunchKernelGGL(split_sum_rope_kernel, dim3(m, (w.rows + 1023) / 1024), dim3(256), 0, s, ws, t.splits, stride,
                           w.rows, ep);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return set_error(SQ_ERR_HIP, std::string("split sum launch: ") + hipGetErrorString(e));
        return 0;
    }
    // where run_rows would pair tiles or split K (other sums than the plain path's)
    if ((gx + 1) / 2 * gy >= device_cus() || (gx * gy < device_cus() && KB / (RW_NW * 2 * RW_NB) >= 2)) return -1;
    count_launch(1, SHAPE_ROWS);
    return launch_rows<WT, 1, RW_QKV>(s, w, aq, ad, m, nullptr, 0, false, gx, gy, 1, KB, nullptr, ep);
}

template <int WT, int NBL, int MT>
int run(hipStream_t s, const MatView& w, const float* x, int m, float* out, int ldo, bool acc) {
    dim3 grid((w.rows + TN - 1) / TN, (m + MT - 1) / MT);
    hipLaunchKernelGGL((gemm_kernel<WT, NBL, MT>), grid, dim3(WAVES * 64), 0, s, w, x, m, out, ldo, acc ? 1 : 0);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return set_error(SQ_ERR_HIP, std::string("gemm launch: ") + hipGetErrorString(e));
    return 0;
}

template <int WT>
int run_f32(hipStream_t s, const MatView& w, const float* x, int m, float* out, int ldo, bool acc) {
    const int KB = w.k / 32;
    if (KB <= 64) return run<WT, 1, 8>(s, w, x, m, out, ldo, acc);
    if (KB <= 256) return run<WT, 4, 2>(s, w, x, m, out, ldo, acc);
    return set_error(SQ_ERR_SHAPE, "gemm: k above 8192 is not supported");
}

}  // namespace

void gemm_counters(bool reset, uint64_t* out) {
    if (out) {
        out[0] = g_launches.load();
        out[1] = g_split_launches.load();
        out[2] = g_shape_launches[SHAPE_128].load();
        out[3] = g_max_splits.load();
        out[4] = g_shape_launches[SHAPE_128X64].load();
        out[5] = g_shape_launches[SHAPE_ROWS].load();
    }
    if (reset) {
        g_launches = 0;
        g_split_launches = 0;
        g_max_splits = 0;
        for (auto& n : g_shape_launches) n = 0;
    }
}

uint64_t gemm_tile64x128_launches() { return g_shape_launches[SHAPE_64X128].load(); }

int launch_gemm_shared(hipStream_t s, const DevMatrix* const* ws, int n, const int8_t* aq, const uint16_t* ad, int m,
                       float* const* outs) {
    if (n < 1 || n > kSharedMax || m <= 0) return -1;
    for (int i = 0; i < n; i++) {
        const DevMatrix& w = *ws[i];
        if (w.fq == nullptr || w.wtype != ws[0]->wtype || w.k != ws[0]->k || w.k <= 0 || w.k % 32 != 0 || w.rows <= 0 ||
            !rows_kernel_fits(m, w.k))
            return -1;
        const RowsPlan p = rows_plan(w, m, true, kGemmSplitFloats);
        if (p.two || p.splits != 1) return -1;
        // outputs that share memory are written in their order, launch by launch
        for (int j = 0; j < i; j++)
            if ((uintptr_t)outs[i] < (uintptr_t)(outs[j] + (size_t)m * ws[j]->rows) &&
                (uintptr_t)outs[j] < (uintptr_t)(outs[i] + (size_t)m * w.rows))
                return -1;
    }
    if (ws[0]->wtype == WT_Q8_0) return run_rows_shared<WT_Q8_0>(s, ws, n, aq, ad, m, outs);
    if (ws[0]->wtype == WT_Q4_0) return run_rows_shared<WT_Q4_0>(s, ws, n, aq, ad, m, outs);
    return -1;
}

int launch_gateup_silu(hipStream_t s, const DevMatrix& w, const int8_t* aq, const uint16_t* ad, int m, int8_t* act_q,
                       uint16_t* act_d, float* ws, size_t ws_floats) {
    if (w.k <= 0 || w.k % 32 != 0 || m <= 0 || w.fq == nullptr) return -1;
    if (w.wtype == WT_Q8_0) return run_gateup_silu<WT_Q8_0>(s, w, aq, ad, m, act_q, act_d, ws, ws_floats);
    if (w.wtype == WT_Q4_0) return run_gateup_silu<WT_Q4_0>(s, w, aq, ad, m, act_q, act_d, ws, ws_floats);
    return -1;
}

int launch_qkv_rope(hipStream_t s, const DevMatrix& w, const int8_t* aq, const uint16_t* ad, int m, int q_dim,
                    int kv_dim, int head_dim, int pos0, const float2* rope, float* q_out, float* kcache, float* vcache,
                    float* ws, size_t ws_floats) {
    if (w.k <= 0 || w.k % 32 != 0 || m <= 0 || w.fq == nullptr) return -1;
    RowsEpi ep{};
    ep.rope = rope;
    ep.q_out = q_out;
    ep.kcache = kcache;
    ep.vcache = vcache;
    ep.q_dim = q_dim;
    ep.kv_dim = kv_dim;
    ep.head_dim = head_dim;
    ep.pos0 = pos0;
    if (w.wtype == WT_Q8_0) return run_qkv_rope<WT_Q8_0>(s, w, aq, ad, m, ep, ws, ws_floats);
    if (w.wtype == WT_Q4_0) return run_qkv_rope<WT_Q4_0>(s, w, aq, ad, m, ep, ws, ws_floats);
    return -1;
}

int launch_gemm(hipStream_t s, const DevMatrix& w, bool a8, const int8_t* aq, const uint16_t* ad, const float* x,
                int m, float* out, int ldo, bool accumulate, float* ws, size_t ws_floats, const NormThen* then) {
    if (w.k <= 0 || w.k % 32 != 0) return set_error(SQ_ERR_SHAPE, "gemm: k must be a positive multiple of 32");
    if (m <= 0) return set_error(SQ_ERR_EMPTY, "gemm: no rows");
    if (w.rows <= 0) return set_error(SQ_ERR_SHAPE, "gemm: the matrix has no rows");
    if (a8 && (w.wtype == WT_Q8_0 || w.wtype == WT_Q4_0)) {
        const int st = w.fq == nullptr
                           ? (w.wtype == WT_Q8_0 ? run_slabs<WT_Q8_0>(s, w, aq, ad, m, out, ldo, accumulate, ws, ws_floats)
                                                 : run_slabs<WT_Q4_0>(s, w, aq, ad, m, out, ldo, accumulate, ws, ws_floats))
                       : w.wtype == WT_Q8_0
                           ? run_integer<WT_Q8_0>(s, w, aq, ad, m, out, ldo, accumulate, ws, ws_floats, &then)
                           : run_integer<WT_Q4_0>(s, w, aq, ad, m, out, ldo, accumulate, ws, ws_floats, &then);
        if (st || !then) return st;
        return launch_rmsnorm_rows(s, out, then->w, m, ldo, then->eps, nullptr, then->act_q, then->act_d);
    }
    switch (w.wtype) {
        case WT_Q8_0:
            return run_f32<WT_Q8_0>(s, view(w), x, m, out, ldo, accumulate);
        case WT_Q4_0:
            return run_f32<WT_Q4_0>(s, view(w), x, m, out, ldo, accumulate);
        case WT_BF16:
            if (a8) return set_error(SQ_ERR_INVALID_TYPE, "gemm: BF16 weights take f32 activations");
            return run_f32<WT_BF16>(s, view(w), x, m, out, ldo, accumulate);
        default:
            return set_error(SQ_ERR_INVALID_TYPE, "gemm: unsupported weight type");
    }
}

}  // namespace sq
