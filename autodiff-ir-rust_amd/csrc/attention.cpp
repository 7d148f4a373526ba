// softmax(scale * Q K^T) V in one kernel, FP32 on the matrix cores: the attention of reference
// src/nn/transformer.rs:10-18 (`dot(softmax(dot(Q, K^T) / sqrt(d_model), -1), V)`), which the reference runs as two
// one-thread-per-element products with the softmax's element-wise and reduction kernels in between, every
// intermediate [Sq, Sk] matrix in memory.  Here the scores never leave the chip.
//
// A block is 4 WG wavefronts on 64 query rows: wavefront w works on rows 16 (w % 4) .. + 15 and, of every tile of BN
// keys, on keys (w / 4) BN / WG .. + BN / WG - 1; with WG = 2 the two halves keep their own running maximum, sum and
// accumulators, which are merged at the end (the same arithmetic as the softmax the caller wrote: exp2((x - max) *
// log2 e), normalised by the sum; accumulators are rescaled when the maximum grows).  K and V tiles live in two LDS
// stages: while one is computed on, the next tile (fetched into registers one iteration earlier) is parked in the
// other, with one barrier per tile.  The probabilities go from the accumulator layout to the operand layout through
// the wavefront's own part of LDS.  Operand reads from LDS run one MFMA step ahead of the MFMAs that use them.
//
// On this hardware FP32 MFMAs and ordinary vector instructions do not overlap (neither within a wavefront nor between
// the wavefronts of a SIMD: a loop of 64 MFMAs and a loop of 512 vector operations take as long together as one after
// the other), so every vector instruction in the loop costs matrix time: addresses are computed once outside the
// loop, ragged-edge masking and the rescaling of the accumulators only run when they are needed.
//
// MFMA 16x16x4 f32: A[i = lane % 16][k = lane / 16], B[k = lane / 16][j = lane % 16], C[4 (lane / 16) + r][lane % 16].
// With D % 16 == 0 the contraction index of the scores is spread over the lanes in runs of four (in step (S, u) lane
// group lq supplies element 16 S + 4 lq + u), so a lane's operands for four consecutive steps are one 128-bit LDS
// read; the weighted values use the same spreading over the keys of a tile.
//
// On the bf16 matrix cores (`parts`: keys of 32, 64, 96 or 128 features, values of 32, 64 or 128, no mask, and as many keys as the
// lowering asks for, at least 32): every FP32 operand as three bf16 parts, as in gemm_split.cpp, with keys and values split and put into the order of the lanes by a kernel of its own before.
// A wavefront owns all 64 query rows and every eighth tile of 32 keys, with its own running maxima, sums and accumulators, so
// that nothing is shared and no barrier stands in the loop; the eight are merged at the end.  It multiplies keys by query
// rows and values by probabilities, so that a row of the softmax is a lane: its maximum takes one exchange between the
// lane's halves, its rescaling none, and the probabilities stand in the registers in which the second product wants them.  What
// does not come out finite -- operands from 2^111 on, infinities, NaN -- is computed again by the kernel described above.
// 8 heads of 2048 x 2048 x 128: 182 us -> 94 and 8 for the split; the matrix instructions take 50, the merging and the first
// trips to memory some 15, and what comes from L2 (0.8 GB) the rest: with 32 query rows a wavefront, twice of that, 98.  With keys and
// values split in the kernel itself, once per row block, it was bound by vector instructions (127 us).  8 heads of 1001 x 1001 x 64:
// 51 -> 24 + 5.  Errors against 64 bits 7.3e-7 -> 5.5e-7 and 4.9e-7 -> 2.4e-7 of a whole attention layer.
#include "attention.hpp"

#include <algorithm>

#include "common.hpp"
#include "gemm.hpp"

namespace adhip {

size_t attention_lds_bytes(const AttentionConfig& cfg) {
    const size_t stage = (size_t)cfg.bn * (size_t)(cfg.d + 4 + cfg.dv + 4);
    const size_t patches = (size_t)4 * cfg.wg * 16 * (size_t)(cfg.bn / cfg.wg + 4);
    const size_t f32 = 4 * (2 * stage + patches);
    if (!cfg.parts) return f32;
    const size_t loop = (size_t)64 * cfg.d * 6, merge = (size_t)4 * 64 * (cfg.dv + 4) * 4;
    return std::max({f32, loop, merge});
}

// 128-bit words of a tile of 32 keys in parts: 16 features of the keys, then 16 keys of the values, 64 lanes and three parts each
static int tile_words(const AttentionConfig& cfg) { return 64 * 3 * (cfg.d / 16 + 2 * (cfg.dv / 32)); }
int64_t attention_parts_floats(const AttentionConfig& cfg, int64_t sk) { return (sk + 31) / 32 * tile_words(cfg) * 4; }

// K and V of every problem in parts, in the order in which the attention kernel's lanes take them: a block does one tile of one
// problem, its wavefronts take turns.  Every row block of a problem would split them again otherwise: 13 vector instructions
// a pair of numbers, 830 of 1180 of a tile, and at five cycles each these, not the matrix instructions, bound the kernel (8 heads
// of 2048 x 2048 x 128: 127 us; 60 and 9 for this pass).
std::string attention_split_source(const AttentionConfig& cfg, const std::string& entry) {
    std::string params, pick;
    for (int i = 0; i < kAttentionSlots; ++i) {
        params += strf("const float* k%d, const float* v%d, ", i, i);
        pick += strf("    case %d: K = k%d; V = v%d; break;\n", i, i, i);
    }
    return strf("#define D %d\n#define DV %d\n#define WORDS %d\n#define EDGE 1\n#define NB (DV / 32)\n#define SCALE 65536.0f\n", cfg.d, cfg.dv, tile_words(cfg)) +
           split_types() + "extern \"C\" __global__ __launch_bounds__(256) void " + entry + "(const int* __restrict__ guard, " + params +
           "float* parts, long long Sk, long long k_ld, long long v_ld) {\n    if (guard && *guard == 0) return;\n    const float* __restrict__ K;\n"
           "    const float* __restrict__ V;\n    switch (blockIdx.y) {\n" + pick + "    default: return;\n    }\n" + R"(
    const unsigned lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, li = lane & 31u, lh = lane >> 5;
    const long long kb = min(32ll * blockIdx.x, Sk - 32);
    uint4_t* to = (uint4_t*)parts + ((long long)blockIdx.y * ((Sk + 31) / 32) + blockIdx.x) * WORDS + lane;
    auto store8 = [&](const float (&x)[8], int unit) {
        uint4_t p0, p1, p2;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            unsigned u0, u1, u2;
            split(x[2 * q], x[2 * q + 1], SCALE, u0, u1, u2);
            p0[q] = u0;
            p1[q] = u1;
            p2[q] = u2;
        }
        to[(3 * unit + 0) * 64] = p0;
        to[(3 * unit + 1) * 64] = p1;
        to[(3 * unit + 2) * 64] = p2;
    };
    for (unsigned u = wave; u < D / 16 + 2; u += 4) {
        if (u < D / 16) {
            // key li, features 16 u + 8 lh ..
            const float* from = K + (kb + li) * k_ld + 16 * u + 8 * lh;
            float x[8];
            *(float4_t*)&x[0] = *(const float4_t*)from;
            *(float4_t*)&x[4] = *(const float4_t*)(from + 4);
            store8(x, u);
        } else {
            // features NB li + i of keys 16 s + 8 (q / 4) + 4 lh + q % 4
            const unsigned s = u - D / 16;
            float v[8][NB];
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const float* from = V + (kb + 16 * s + 8 * (q >> 2) + 4 * lh + (q & 3)) * v_ld + NB * li;
#if NB == 4
                *(float4_t*)v[q] = *(const float4_t*)from;
#elif NB == 2
                *(float2_t*)v[q] = *(const float2_t*)from;
#else
                v[q][0] = *from;
#endif
            }
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                float x[8];
#pragma unroll
                for (int q = 0; q < 8; ++q) x[q] = v[q][i];
                store8(x, D / 16 + s * NB + i);
            }
        }
    }
}
)";
}

std::string attention_kernel_source(const AttentionConfig& cfg, const std::string& entry) {
    ADHIP_CHECK(!cfg.parts || (!cfg.mask && cfg.wg == 2 && attention_takes_parts(cfg.d, cfg.dv)), "internal: attention of these widths in bf16 parts");
    std::string s;
    std::string params, pick = "switch (problem) {";
    for (int i = 0; i < kAttentionSlots; ++i) {
        params += strf("float* o%d, const float* q%d, const float* k%d, const float* v%d, ", i, i, i, i);
        if (cfg.mask) params += strf("const float* m%d, ", i);
        pick += strf(" case %d: O = o%d; Q = q%d; K = k%d; V = v%d;%s break;", i, i, i, i, i, cfg.mask ? strf(" Mk = m%d;", i).c_str() : "");
    }
    s += "#define GROUP_PARAMS " + params + "\n#define GROUP_PICK " + pick + " default: return; }\n";
    s += strf("#define KERNEL_NAME %s\n#define D %d\n#define DV %d\n#define BN %d\n#define WG %d\n#define MASK %d\n#define PARTS %d\n#define LDS_FLOATS %zu\n#define WORDS %d\n", entry.c_str(), cfg.d, cfg.dv, cfg.bn,
              cfg.wg, cfg.mask ? 1 : 0, cfg.parts ? 1 : 0, attention_lds_bytes(cfg) / 4, cfg.parts ? tile_words(cfg) : 0);
    s += cfg.parts ? "#define PARTS_POINTER const float* __restrict__ parts,\n" : "#define PARTS_POINTER\n";
    s += cfg.mask ? "#define MASK_LD long long m_ld,\n" : "#define MASK_LD\n";
    if (cfg.parts) s += "#define EDGE 1\n" + split_types();
    else
        s += "typedef float float4_t __attribute__((ext_vector_type(4)));\n";
    s += R"ATTN(
#define NT (256 * WG)
#define BNW (BN / WG)
#define KLD (D + 4)
#define VLD (DV + 4)
#define PLD (BNW + 4)
#define STAGE (BN * KLD + BN * VLD)
// Value of lane (16 q + perm(i)) for every lane 16 q + i; every lane has a source, so the "old" value never shows.
#define ROW16_FROM(x, ctrl) __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, (x)), (ctrl), 0xF, 0xF, true))
static __device__ __forceinline__ float row16_max(float x) {
    // maximum over the 16 lanes that share an accumulator row (lanes 16 q .. 16 q + 15)
    x = fmaxf(x, ROW16_FROM(x, 0xB1));    // quad_perm [1,0,3,2]
    x = fmaxf(x, ROW16_FROM(x, 0x4E));    // quad_perm [2,3,0,1]
    x = fmaxf(x, ROW16_FROM(x, 0x141));   // row_half_mirror
    x = fmaxf(x, ROW16_FROM(x, 0x140));   // row_mirror
    return x;
}
static __device__ __forceinline__ float row16_sum(float x) {
    // every step adds a lane's value and its partner's, both partners in the same way: all 16 lanes end with the same bits
    x += ROW16_FROM(x, 0xB1);
    x += ROW16_FROM(x, 0x4E);
    x += ROW16_FROM(x, 0x141);
    x += ROW16_FROM(x, 0x140);
    return x;
}

extern "C" __global__ __launch_bounds__(NT) void KERNEL_NAME(
    const int* __restrict__ guard, GROUP_PARAMS PARTS_POINTER long long Sq, long long Sk, long long q_ld, long long k_ld, long long v_ld,
    MASK_LD float scale, int row_blocks, int problems) {
    if (guard && *guard == 0) return;
    // Blocks are handed to the eight XCDs in turn; renumbering them so that an XCD's blocks are consecutive puts the row
    // blocks of one problem on one XCD, whose L2 then fetches that problem's K and V once.
    unsigned bid = blockIdx.x;
    {
        const unsigned total = (unsigned)row_blocks * (unsigned)problems;
        if (total % 8u == 0u) bid = (bid % 8u) * (total / 8u) + bid / 8u;
    }
    const unsigned problem = bid / (unsigned)row_blocks, row_block = bid % (unsigned)row_blocks;
    float* __restrict__ O;
    const float* __restrict__ Q;
    const float* __restrict__ K;
    const float* __restrict__ V;
#if MASK
    const float* __restrict__ Mk;
#endif
    GROUP_PICK
    __shared__ __attribute__((aligned(16))) float lds[LDS_FLOATS];
    const float LOG2E = 1.44269502162933349609375f;  // the float nearest 1 / ln 2
    const unsigned tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
#if PARTS
#define SCALE 65536.0f
#define NB (DV / 32)                    /* blocks of 32 features of the result */
    {
        __shared__ int failed;
        const unsigned li = lane & 31u, lh = lane >> 5, kg = __builtin_amdgcn_readfirstlane(wave);
        const long long row0 = (long long)row_block * 64;
        // the block's query rows in parts: [part][eight features][row]
        uint4_t* Qs = (uint4_t*)lds;
#pragma unroll
        for (unsigned u0 = 0; u0 < 64 * D / 8; u0 += NT) {
            const unsigned u = u0 + tid, row = u / (D / 8), d8 = u % (D / 8);
            if (64 * D / 8 % NT == 0 || u < 64 * D / 8) {
                const float* from = Q + min(row0 + (long long)row, Sq - 1) * q_ld + 8 * d8;
                float x[8];
                *(float4_t*)&x[0] = *(const float4_t*)from;
                *(float4_t*)&x[4] = *(const float4_t*)(from + 4);
                uint4_t p0, p1, p2;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    unsigned u0, u1, u2;
                    split(x[2 * q], x[2 * q + 1], SCALE, u0, u1, u2);
                    p0[q] = u0;
                    p1[q] = u1;
                    p2[q] = u2;
                }
                Qs[(0 * (D / 8) + d8) * 64 + row] = p0;
                Qs[(1 * (D / 8) + d8) * 64 + row] = p1;
                Qs[(2 * (D / 8) + d8) * 64 + row] = p2;
            }
        }
        // Keys and values come in parts and in the order of the lanes (see the kernel that splits them): a unit is what six
        // matrix instructions take of them, first 16 features of the 32 keys at a time, then 16 keys of 32 features of the values
        // at a time.  Two to four units are on their way; behind its last tile a wavefront fetches the last unit once more.
#define UNITS (D / 16 + 2 * NB)
#define RING (NB == 4 ? 2 : UNITS % 4 == 0 ? 4 : UNITS % 3 == 0 ? 3 : 2)
        const uint4_t* from = (const uint4_t*)parts + (long long)problem * ((Sk + 31) / 32) * WORDS;
        const unsigned lane_at = 16u * lane;
        uint4_t ring[RING][3];
        auto fetch = [&](long long t, int unit) {
#pragma unroll
            for (int p = 0; p < 3; ++p) ring[unit % RING][p] = *(const uint4_t*)((const char*)(from + t * WORDS + (3 * unit + p) * 64) + lane_at);
        };
        auto split8 = [&](const float (&x)[8], float scale, bf16x8_t (&p)[3]) {
            uint4_t a, b, c;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                unsigned u0, u1, u2;
                split(x[2 * q], x[2 * q + 1], scale, u0, u1, u2);
                a[q] = u0;
                b[q] = u1;
                c[q] = u2;
            }
            p[0] = __builtin_bit_cast(bf16x8_t, a);
            p[1] = __builtin_bit_cast(bf16x8_t, b);
            p[2] = __builtin_bit_cast(bf16x8_t, c);
        };
        // of the nine products of parts the six that reach the result's 24 bits, the smallest first
#define TERM(acc, x, y)                                                                                                  \
        acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x, y[0], acc[0], 0, 0, 0);                                     \
        acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x, y[1], acc[1], 0, 0, 0);
#define SIX(acc, x, y)                                                                                                   \
        TERM(acc, x[2], y[0]) TERM(acc, x[0], y[2]) TERM(acc, x[1], y[1]) TERM(acc, x[1], y[0]) TERM(acc, x[0], y[1]) TERM(acc, x[0], y[0])
        float16_t o[NB][2];   // o[i][j][4 g + r]: feature NB (8 g + 4 lh + r) + i of query row 32 j + li
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) o[i][0][r] = o[i][1][r] = 0.0f;
        float m[2] = {-__builtin_inff(), -__builtin_inff()}, l[2] = {0.0f, 0.0f};   // of query row 32 j + li; the sum over this half's keys
        const float unscale = scale * (1.0f / SCALE / SCALE);
        // the matrix cores lose a little towards minus infinity: every other key group weighs with the other sign
        const float p_scale = kg & 1u ? -SCALE : SCALE;
        const long long tiles = (Sk + 31) / 32;
        if (kg < tiles) {
#pragma unroll
            for (int u = 0; u < RING; ++u) fetch(kg, u);
        }
        __syncthreads();
#pragma unroll 1
        for (long long t = kg; t < tiles; t += 8) {
            const long long t_next = t + 8 < tiles ? t + 8 : t;
            bf16x8_t f[3];
            auto next = [&](int unit) {   // takes a unit and asks for the one that will stand in its place
#pragma unroll
                for (int p = 0; p < 3; ++p) f[p] = __builtin_bit_cast(bf16x8_t, ring[unit % RING][p]);
                if (unit + RING < UNITS) fetch(t, unit + RING);
                else fetch(t_next, unit + RING - UNITS);
            };
            // scores, keys by query rows
            float16_t sc[2];
#pragma unroll
            for (int r = 0; r < 16; ++r) sc[0][r] = sc[1][r] = 0.0f;
#pragma unroll
            for (int u = 0; u < D / 16; ++u) {
                bf16x8_t qf[3][2];
#pragma unroll
                for (int p = 0; p < 3; ++p)
#pragma unroll
                    for (int j = 0; j < 2; ++j) qf[p][j] = __builtin_bit_cast(bf16x8_t, Qs[(p * (D / 8) + 2 * u + lh) * 64 + 32 * j + li]);
                next(u);
                SIX(sc, f, qf)
                __builtin_amdgcn_sched_barrier(0);   // (operands of later units taken from LDS now are registers that a wide head lacks)
            }
            if (32 * t + 32 > Sk) {   // the last tile begins earlier, with keys that the tile before has
                const int had = (int)(32 * t + 32 - Sk);
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    if (8 * (r >> 2) + 4 * (int)lh + (r & 3) < had) sc[0][r] = sc[1][r] = -__builtin_inff();
            }
            float m_new[2];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                float mx = -__builtin_inff();
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    sc[j][r] *= unscale;
                    mx = fmaxf(mx, sc[j][r]);
                }
                m_new[j] = fmaxf(m[j], fmaxf(mx, __shfl_xor(mx, 32)));
            }
            if (__builtin_amdgcn_ballot_w64(m_new[0] != m[0] || m_new[1] != m[1]) != 0ull) {
                // some row's maximum grew: what has been accumulated against the old maximum is rescaled
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const float alpha = __builtin_amdgcn_exp2f((m[j] - m_new[j]) * LOG2E);
                    l[j] *= alpha;
#pragma unroll
                    for (int i = 0; i < NB; ++i)
#pragma unroll
                        for (int r = 0; r < 16; ++r) o[i][j][r] *= alpha;
                    m[j] = m_new[j];
                }
            }
            // probabilities stand as the second product wants them: a lane's keys are its keys again
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                bf16x8_t pf[3][2];
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    float p[8];
                    bf16x8_t parts_of_p[3];
#pragma unroll
                    for (int q = 0; q < 8; ++q) {
                        p[q] = __builtin_amdgcn_exp2f((sc[j][4 * (2 * s + (q >> 2)) + (q & 3)] - m[j]) * LOG2E);
                        l[j] += p[q];
                    }
                    split8(p, p_scale, parts_of_p);
#pragma unroll
                    for (int x = 0; x < 3; ++x) pf[x][j] = parts_of_p[x];
                }
#pragma unroll
                for (int i = 0; i < NB; ++i) {
                    next(D / 16 + s * NB + i);
                    SIX(o[i], f, pf)
                }
            }
        }
        // half of the key groups hand theirs to the other half, three times
#pragma unroll
        for (int half = 4; half >= 1; half >>= 1) {
            __syncthreads();
            float* mg = lds + (kg & (half - 1)) * 64 * (32 * NB + 4) + lane * (32 * NB + 4);
            if ((int)kg >= half && (int)kg < 2 * half) {
                *(float4_t*)mg = float4_t{m[0], m[1], l[0], l[1]};
#pragma unroll
                for (int i = 0; i < NB; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j)
#pragma unroll
                        for (int g = 0; g < 4; ++g)
                            *(float4_t*)(mg + 4 + 32 * i + 16 * j + 4 * g) = float4_t{o[i][j][4 * g], o[i][j][4 * g + 1], o[i][j][4 * g + 2], o[i][j][4 * g + 3]};
            }
            __syncthreads();
            if ((int)kg < half) {
                const float4_t theirs = *(const float4_t*)mg;
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    // (a group without keys has -inf and zeros; one in front of a group with keys has keys)
                    const float top = fmaxf(m[j], theirs[j]);
                    const float e0 = m[j] == top ? 1.0f : __builtin_amdgcn_exp2f((m[j] - top) * LOG2E);
                    const float e1 = theirs[j] == -__builtin_inff() ? 0.0f : __builtin_amdgcn_exp2f((theirs[j] - top) * LOG2E);
                    // groups of odd number have the other sign: all of the first round's pairs agree, and so do the second's
                    const float es = half == 1 ? -e1 : e1;
                    l[j] = l[j] * e0 + theirs[2 + j] * e1;
                    m[j] = top;
#pragma unroll
                    for (int i = 0; i < NB; ++i)
#pragma unroll
                        for (int g = 0; g < 4; ++g) {
                            const float4_t v = *(const float4_t*)(mg + 4 + 32 * i + 16 * j + 4 * g);
#pragma unroll
                            for (int r = 0; r < 4; ++r) o[i][j][4 * g + r] = o[i][j][4 * g + r] * e0 + v[r] * es;
                        }
                }
            }
        }
        if (kg == 0) {
            unsigned largest = 0u;
            float inv[2];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                l[j] += __shfl_xor(l[j], 32);
                inv[j] = (1.0f / l[j]) * (1.0f / SCALE / SCALE);
                largest = max(largest, __builtin_bit_cast(unsigned, l[j]) & 0x7fffffffu);
#pragma unroll
                for (int i = 0; i < NB; ++i)
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const float x = o[i][j][r];
                        largest = max(largest, __builtin_bit_cast(unsigned, x) & 0x7fffffffu);
                    }
            }
            const bool bad = __builtin_amdgcn_ballot_w64(largest >= 0x7f800000u) != 0ull;
            if (lane == 0) failed = bad;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const long long row = row0 + 32 * j + li;
                if (!bad && row < Sq) {
#pragma unroll
                    for (int g = 0; g < 4; ++g)
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            float* to = O + row * DV + NB * (8 * g + 4 * lh + r);
#if NB == 4
                            *(float4_t*)to = float4_t{o[0][j][4 * g + r], o[1][j][4 * g + r], o[NB - 2][j][4 * g + r], o[NB - 1][j][4 * g + r]} * inv[j];
#else
#pragma unroll
                            for (int i = 0; i < NB; ++i) to[i] = o[i][j][4 * g + r] * inv[j];
#endif
                        }
                }
            }
        }
        __syncthreads();
        if (!failed) return;
        __syncthreads();
    }
#endif
    float (*Ps)[16][PLD] = (float (*)[16][PLD])(lds + 2 * STAGE);
    const unsigned li = lane & 15u, lq = lane >> 4, rw = wave & 3u, kg = wave >> 2;
    const long long row_base = (long long)row_block * 64 + rw * 16;

    // this lane's part of the wavefront's 16 query rows
#if D % 16 == 0
    float4_t qf[D / 16];
    {
        const long long row = row_base + li;
#pragma unroll
        for (int S = 0; S < D / 16; ++S)
            qf[S] = row < Sq ? *(const float4_t*)(Q + row * q_ld + 16 * S + 4 * lq) : float4_t{0.f, 0.f, 0.f, 0.f};
    }
#else
    float qf[D / 4];
    {
        const long long row = row_base + li;
#pragma unroll
        for (int s = 0; s < D / 4; ++s) qf[s] = row < Sq ? Q[row * q_ld + 4 * s + lq] : 0.0f;
    }
#endif
    float4_t oacc[DV / 16];
#pragma unroll
    for (int nb = 0; nb < DV / 16; ++nb) oacc[nb] = float4_t{0.f, 0.f, 0.f, 0.f};
    float m_i[4], l_i[4];   // running maximum of the row; this lane's share of the running sum (added up at the end)
#pragma unroll
    for (int r = 0; r < 4; ++r) { m_i[r] = -__builtin_inff(); l_i[r] = 0.0f; }
#if MASK
    // where this lane's four accumulator rows start in the mask, at this key group's and lane's column (rows beyond Sq
    // are never stored: they read the last row)
    const float* mrow[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const long long row = row_base + 4 * lq + r;
        mrow[r] = Mk + (row < Sq ? row : Sq - 1) * m_ld + kg * BNW + li;
    }
#endif

    // The next tile travels through registers.  Where a thread's pieces sit inside a tile, in memory and in LDS, is
    // computed once; a tile's base is uniform.  Keys beyond Sk (last tile only) are fetched from the last valid row
    // instead: their scores are masked to -inf and their probabilities are 0, so what stands there only has to be finite.
    constexpr int KL = (BN * D / 4 + NT - 1) / NT, VL = (BN * DV / 4 + NT - 1) / NT;
    float4_t kr[KL], vr[VL];
    unsigned k_key[KL], k_mem[KL], k_lds[KL], v_key[VL], v_mem[VL], v_lds[VL];
#pragma unroll
    for (int i = 0; i < KL; ++i) {
        const unsigned idx = tid + NT * i, key = idx / (D / 4), f4 = idx % (D / 4);
        k_key[i] = key; k_mem[i] = key * (unsigned)k_ld + 4 * f4; k_lds[i] = key * KLD + 4 * f4;
    }
#pragma unroll
    for (int i = 0; i < VL; ++i) {
        const unsigned idx = tid + NT * i, key = idx / (DV / 4), f4 = idx % (DV / 4);
        v_key[i] = key; v_mem[i] = key * (unsigned)v_ld + 4 * f4; v_lds[i] = BN * KLD + key * VLD + 4 * f4;
    }
    auto fetch = [&](long long k0) {
        const float* kb = K + k0 * k_ld;
        const float* vb = V + k0 * v_ld;
        if (k0 + BN <= Sk) {
#pragma unroll
            for (int i = 0; i < KL; ++i)
                if (BN * D / 4 % NT == 0 || tid + NT * i < BN * D / 4) kr[i] = *(const float4_t*)(kb + k_mem[i]);
#pragma unroll
            for (int i = 0; i < VL; ++i)
                if (BN * DV / 4 % NT == 0 || tid + NT * i < BN * DV / 4) vr[i] = *(const float4_t*)(vb + v_mem[i]);
        } else {
            const unsigned last = (unsigned)(Sk - 1 - k0);
#pragma unroll
            for (int i = 0; i < KL; ++i)
                if (BN * D / 4 % NT == 0 || tid + NT * i < BN * D / 4) {
                    const unsigned back = k_key[i] > last ? k_key[i] - last : 0u;
                    kr[i] = *(const float4_t*)(kb + (k_mem[i] - back * (unsigned)k_ld));
                }
#pragma unroll
            for (int i = 0; i < VL; ++i)
                if (BN * DV / 4 % NT == 0 || tid + NT * i < BN * DV / 4) {
                    const unsigned back = v_key[i] > last ? v_key[i] - last : 0u;
                    vr[i] = *(const float4_t*)(vb + (v_mem[i] - back * (unsigned)v_ld));
                }
        }
    };
    auto park = [&](int stage) {
        float* base = lds + stage * STAGE;
#pragma unroll
        for (int i = 0; i < KL; ++i)
            if (BN * D / 4 % NT == 0 || tid + NT * i < BN * D / 4) *(float4_t*)(base + k_lds[i]) = kr[i];
#pragma unroll
        for (int i = 0; i < VL; ++i)
            if (BN * DV / 4 % NT == 0 || tid + NT * i < BN * DV / 4) *(float4_t*)(base + v_lds[i]) = vr[i];
    };
    fetch(0);
    park(0);
    if (BN < Sk) fetch(BN);
    int stage = 0;
    for (long long k0 = 0; k0 < Sk; k0 += BN, stage ^= 1) {
        // tile k0 is complete in this stage, and everybody is done with the other stage (the previous tile)
        __syncthreads();
        float (*Ks)[KLD] = (float (*)[KLD])(lds + stage * STAGE + kg * BNW * KLD);
        float (*Vs)[VLD] = (float (*)[VLD])(lds + stage * STAGE + BN * KLD + kg * BNW * VLD);
        if (k0 + BN < Sk) {
            park(stage ^ 1);
            if (k0 + 2 * BN < Sk) fetch(k0 + 2 * BN);
        }

        // ---- scores of 16 rows x BNW keys.  The K operands of step S + 1 are read while the MFMAs of step S run;
        // two accumulators per block of 16 keys (even and odd u) keep dependent MFMAs apart.
        float4_t sacc[BNW / 16], sodd[BNW / 16];
#pragma unroll
        for (int nb = 0; nb < BNW / 16; ++nb) { sacc[nb] = float4_t{0.f, 0.f, 0.f, 0.f}; sodd[nb] = float4_t{0.f, 0.f, 0.f, 0.f}; }
#if D % 16 == 0
        {
            float4_t kf[2][BNW / 16];
#pragma unroll
            for (int nb = 0; nb < BNW / 16; ++nb) kf[0][nb] = *(const float4_t*)&Ks[16 * nb + li][4 * lq];
#pragma unroll
            for (int S = 0; S < D / 16; ++S) {
                if (S + 1 < D / 16) {
#pragma unroll
                    for (int nb = 0; nb < BNW / 16; ++nb)
                        kf[(S + 1) & 1][nb] = *(const float4_t*)&Ks[16 * nb + li][16 * (S + 1) + 4 * lq];
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int u = 0; u < 4; u += 2) {
#pragma unroll
                    for (int nb = 0; nb < BNW / 16; ++nb)
                        sacc[nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(qf[S][u], kf[S & 1][nb][u], sacc[nb], 0, 0, 0);
#pragma unroll
                    for (int nb = 0; nb < BNW / 16; ++nb)
                        sodd[nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(qf[S][u + 1], kf[S & 1][nb][u + 1], sodd[nb], 0, 0, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
#else
#pragma unroll
        for (int s = 0; s < D / 4; ++s) {
#pragma unroll
            for (int nb = 0; nb < BNW / 16; ++nb) {
                if (s & 1) sodd[nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(qf[s], Ks[16 * nb + li][4 * s + lq], sodd[nb], 0, 0, 0);
                else sacc[nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(qf[s], Ks[16 * nb + li][4 * s + lq], sacc[nb], 0, 0, 0);
            }
        }
#endif
        // ---- running maximum of every row (rows 4 lq + r of this wavefront; 16 lanes share a row)
        float mx[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) mx[r] = -__builtin_inff();
#if MASK
#pragma unroll
        for (int nb = 0; nb < BNW / 16; ++nb) {
            // the scaled score times the mask, in that order, as the caller wrote it; keys beyond Sk read nothing
            const bool inside = k0 + BN <= Sk || k0 + kg * BNW + 16 * nb + li < Sk;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float mv = inside ? mrow[r][k0 + 16 * nb] : 0.0f;
                sacc[nb][r] = ((sacc[nb][r] + sodd[nb][r]) * scale) * mv;
            }
        }
#else
#pragma unroll
        for (int nb = 0; nb < BNW / 16; ++nb)
#pragma unroll
            for (int r = 0; r < 4; ++r) sacc[nb][r] = (sacc[nb][r] + sodd[nb][r]) * scale;
#endif
        if (k0 + BN > Sk) {   // the last tile may reach beyond the keys
#pragma unroll
            for (int nb = 0; nb < BNW / 16; ++nb) {
                const bool valid = k0 + kg * BNW + 16 * nb + li < Sk;
#pragma unroll
                for (int r = 0; r < 4; ++r) sacc[nb][r] = valid ? sacc[nb][r] : -__builtin_inff();
            }
        }
#pragma unroll
        for (int nb = 0; nb < BNW / 16; ++nb)
#pragma unroll
            for (int r = 0; r < 4; ++r) mx[r] = fmaxf(mx[r], sacc[nb][r]);
        float m_new[4], mu[4];
        bool grew = false;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            m_new[r] = fmaxf(m_i[r], row16_max(mx[r]));
            grew = grew || m_new[r] != m_i[r];
            // a key group that has not seen a valid key yet keeps -inf; the exponentials are then taken against 0
            mu[r] = m_new[r] == -__builtin_inff() ? 0.0f : m_new[r];
        }
        if (__builtin_amdgcn_ballot_w64(grew) != 0ull) {
            // some row's maximum grew: what has been accumulated against the old maximum is rescaled
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float alpha = __builtin_amdgcn_exp2f((m_i[r] - mu[r]) * LOG2E);
                l_i[r] *= alpha;
#pragma unroll
                for (int nb = 0; nb < DV / 16; ++nb) oacc[nb][r] *= alpha;
                m_i[r] = m_new[r];
            }
        }
#pragma unroll
        for (int nb = 0; nb < BNW / 16; ++nb) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float p = __builtin_amdgcn_exp2f((sacc[nb][r] - mu[r]) * LOG2E);
                l_i[r] += p;
                Ps[wave][4 * lq + r][16 * nb + li] = p;
            }
        }
        // the probabilities go from the accumulator layout to the operand layout through this wavefront's own part of
        // LDS; a wavefront's LDS accesses are carried out in order, the compiler only has to keep them in order too
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        {
            // ---- weighted values: step t covers four keys of this wavefront's share (in the spread order); the V
            // operands of step t + 1 are read while the MFMAs of step t run
            float4_t a[BNW / 16];
#pragma unroll
            for (int S = 0; S < BNW / 16; ++S) a[S] = *(const float4_t*)&Ps[wave][li][16 * S + 4 * lq];
            float vb[2][DV / 16];
#pragma unroll
            for (int nb = 0; nb < DV / 16; ++nb) vb[0][nb] = Vs[4 * lq][16 * nb + li];
#pragma unroll
            for (int t = 0; t < BNW / 4; ++t) {
                if (t + 1 < BNW / 4) {
#pragma unroll
                    for (int nb = 0; nb < DV / 16; ++nb)
                        vb[(t + 1) & 1][nb] = Vs[16 * ((t + 1) / 4) + 4 * lq + ((t + 1) & 3)][16 * nb + li];
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int nb = 0; nb < DV / 16; ++nb)
                    oacc[nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[t / 4][t & 3], vb[t & 1][nb], oacc[nb], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) l_i[r] = row16_sum(l_i[r]);
#if WG == 2
    // the second key group hands its maximum, sum and accumulators to the first through LDS (the tiles are done with)
    __syncthreads();
    {
        float* mg = lds + (size_t)(rw * 64 + lane) * (DV / 4 + 8);
        if (kg == 1) {
#pragma unroll
            for (int r = 0; r < 4; ++r) { mg[r] = m_i[r]; mg[4 + r] = l_i[r]; }
#pragma unroll
            for (int nb = 0; nb < DV / 16; ++nb) *(float4_t*)(mg + 8 + 4 * nb) = oacc[nb];
        }
        __syncthreads();
        if (kg == 1) return;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float mb = mg[r], lb = mg[4 + r];
            const float m = fmaxf(m_i[r], mb);   // the first group always holds key 0: finite; a group without keys has -inf and sum 0
            const float ea = __builtin_amdgcn_exp2f((m_i[r] - m) * LOG2E), eb = __builtin_amdgcn_exp2f((mb - m) * LOG2E);
            l_i[r] = l_i[r] * ea + lb * eb;
#pragma unroll
            for (int nb = 0; nb < DV / 16; ++nb) oacc[nb][r] = oacc[nb][r] * ea + mg[8 + 4 * nb + r] * eb;
        }
    }
#endif
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const long long row = row_base + 4 * lq + r;
        const float inv = 1.0f / l_i[r];
        if (row < Sq) {
#pragma unroll
            for (int nb = 0; nb < DV / 16; ++nb) O[row * DV + 16 * nb + li] = oacc[nb][r] * inv;
        }
    }
}
)ATTN";
    return s;
}

}  // namespace adhip
