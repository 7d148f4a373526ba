// FP32 matrix product for gfx950 on the bf16 matrix cores (v_mfma_f32_32x32x16_bf16), LDS-tiled.
//
// An FP32 number times 2^16 is exactly the sum of three bf16 ones (8 + 8 + 8 bits, each rounded to nearest; without the
// factor the last of them would fall below bf16's range where the number is below 2^-110), so a product of two is nine
// products of parts, each exact in FP32 (the method: Henry, Tang, Heinecke, "Leveraging the bfloat16 Artificial
// Intelligence Datatype For Higher-Precision Computations", ARITH 2019).  The six with a weight of 2^-16 and more are
// summed, smallest first, and the sum is taken back by 2^-32; the three left out come to some 2^-27 of the product, a
// fraction of the rounding of one FP32 addition.  A step of 16 k costs 6 x 32 matrix cycles per 32 x 32 block where the
// FP32 matrix cores take 512, and, other than theirs, vector instructions of one wavefront run under the matrix
// instructions of another: the bound is the bf16 matrix rate over six (2.0 PFLOP/s sustained: 330 TFLOP/s).  The matrix
// cores are busy 62-78 % of the time at 4096^3; the splitting takes a quarter of the vector pipes' and the parts a fifth
// of the LDS's, and the rest is time in which no wavefront of a SIMD multiplies.  The sums are rounded twice per 8 k and
// product instead of once per k: errors against 64 bits are no larger (normal operands, k = 4096: 1.0e-6 against 1.1e-6 of
// the root mean square; k = 1024:
// 3.4-4.8e-7 against 5.8e-7; k = 64: 0.7e-7 against 1.4e-7).
//
// The operands are described by strides and split on their way from registers to LDS, where a part's eight consecutive
// k of a row are one 128-bit word, which is what a lane feeds to the matrix instruction.  Tiles, and 4096^3 on each of
// the large ones (FP32 matrix cores, 256x128: 1090 us, 126 TFLOP/s):
//   256x256x16  8 wavefronts of 128x64 in two sets that take turns between multiplying and everything else: 600-650 us
//   128x128x16  4 wavefronts of 64x64, two blocks per CU: 710-770 us
//   128x128x32  8 wavefronts, two per 64x64 sub-tile with half of the k-tile each: one block per CU does what two of
//               the former do (4096 x 1024 x 4096: 181-188 us against 326 on 128x64 FP32 tiles)
//   128x64x32, 64x64x32, 64x64x64 (two sets): outputs of a few hundred blocks with a short k, or a long one in ranges (other
//               small ones: gemm_direct.cpp)
// Ragged sizes cost little: rows beyond the product repeat its last row, and the last k-tile starts inside the one
// before it, with zeros for the k it shares (4000 x 4011 x 4001: 615-665 us against 1567).
#include "gemm.hpp"

#include "common.hpp"

namespace adhip {

std::string split_types() {
    return R"(typedef float float4_t __attribute__((ext_vector_type(4)));
typedef float float2_t __attribute__((ext_vector_type(2)));
typedef float float16_t __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef unsigned uint4_t __attribute__((ext_vector_type(4)));
#if EDGE
#define UNALIGNED __attribute__((aligned(4)))
#else
#define UNALIGNED
#endif
typedef float4_t float4_g UNALIGNED;


// Two neighbours of an operand, times scale (2^16 or -2^16), as three pairs of bf16 whose sums are exactly the two: the
// last bit of the smallest FP32 number, 2^-149, becomes the last bit of the smallest bf16 one.  (Without the factor the
// products take 0-4 % less, 4096 x 1024 x 4096 180.6 us for 184.5, and are wrong for operands below 2^-110.)
static __device__ __forceinline__ unsigned pack(float x, float y) {
    return __builtin_bit_cast(unsigned, __builtin_convertvector((float2_t{x, y}), bf16x2_t));
}
// part p (0, 1, 2 in turn) of two neighbours, which become what is left of them
static __device__ __forceinline__ unsigned split_part(int p, float& x, float& y, float scale) {
    const unsigned u = p == 0 ? pack(x * scale, y * scale) : pack(x, y);
    if (p == 2) return u;
    x = __builtin_fmaf(x, p == 0 ? scale : 1.0f, -__builtin_bit_cast(float, u << 16));
    y = __builtin_fmaf(y, p == 0 ? scale : 1.0f, -__builtin_bit_cast(float, u & 0xffff0000u));
    return u;
}
static __device__ __forceinline__ void split(float x, float y, float scale, unsigned& p0, unsigned& p1, unsigned& p2) {
    p0 = split_part(0, x, y, scale);
    p1 = split_part(1, x, y, scale);
    p2 = split_part(2, x, y, scale);
}

)";
}

std::string split_tail() {
    return R"(    // What the parts cannot represent -- infinities, NaN, operands from 2^111 and sums from 2^95 on -- ends in a sum that
    // is not finite: such a wavefront's sub-tile is multiplied again on the FP32 matrix cores, straight from memory.  A
    // lane takes four consecutive k at a time, and two rows of blocks share what is loaded (all four at once spill):
    // 4096^3 with an infinity in every wavefront's rows 1.8-2.2 ms in all, where one k and one row at a time took 3.8-5.9
    // (FP32 matrix cores alone, staged through LDS: 1.1).
    unsigned largest = 0u;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const float x = acc[i][j][r];   // (a bit cast of a vector's element itself reads the vector's first)
                largest = max(largest, __builtin_bit_cast(unsigned, x) & 0x7fffffffu);
            }
    const bool again_f32 = __builtin_amdgcn_ballot_w64(largest >= 0x7f800000u) != 0ull;
    const float unscale = again_f32 ? 1.0f : 1.0f / SCALE / SCALE;
#define ROWS (TM < 2 ? TM : 2)
#define KEEP(x) asm volatile("" : "+v"(x));   /* step by step: the addresses of all steps at once cost the 256x256 tile its last registers */
#pragma unroll
    for (int i0 = 0; i0 < TM; i0 += ROWS) {
        if (again_f32) {
            long long qa[ROWS], qb[TN];   // where its next four k begin
#pragma unroll
            for (int i = 0; i < ROWS; ++i) {
                qa[i] = CLAMP_A(wm * (32 * TM) + 32 * (i0 + i) + li) * a_sm + (k_lo + 4 * lh) * a_sk;
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) acc[i0 + i][j][r] = 0.0f;
            }
#pragma unroll
            for (int j = 0; j < TN; ++j) qb[j] = CLAMP_B(wn * (32 * TN) + 32 * j + li) * b_sn + (k_lo + 4 * lh) * b_sk;
            auto multiply_f32 = [&](const float* x, const float* y, int stride) {   // one k of a lane
#pragma unroll
                for (int i = 0; i < ROWS; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j)
                        acc[i0 + i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(x[i * stride], y[j * stride], acc[i0 + i][j], 0, 0, 0);
            };
            long long k0 = k_lo;
#pragma unroll 1
            for (; k0 + 8 <= k_hi; k0 += 8) {
                float x[ROWS][4], y[TN][4];
#if A_KCONTIG
#pragma unroll
                for (int i = 0; i < ROWS; ++i) {
                    *(float4_t*)x[i] = *(const float4_g*)(A + qa[i]);
                    qa[i] += 8;
                }
#else
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int i = 0; i < ROWS; ++i) {
                        x[i][q] = A[qa[i]];
                        qa[i] += (q < 3 ? 1 : 5) * a_sk;
                        KEEP(qa[i])
                    }
#endif
#if B_KCONTIG
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    *(float4_t*)y[j] = *(const float4_g*)(B + qb[j]);
                    qb[j] += 8;
                }
#else
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int j = 0; j < TN; ++j) {
                        y[j][q] = B[qb[j]];
                        qb[j] += (q < 3 ? 1 : 5) * b_sk;
                        KEEP(qb[j])
                    }
#endif
#pragma unroll
                for (int q = 0; q < 4; ++q) multiply_f32(&x[0][q], &y[0][q], 4);
            }
#pragma unroll 1
            for (int q = 0; q < 4 && k0 + q < k_hi; ++q) {
                const bool in = k0 + 4 * lh + q < k_hi;   // (beyond: the last k again, as zero)
                const long long at = in ? q : k_hi - 1 - (k0 + 4 * lh);
                float x[ROWS], y[TN];
#pragma unroll
                for (int i = 0; i < ROWS; ++i) x[i] = in ? A[qa[i] + at * a_sk] : 0.0f;
#pragma unroll
                for (int j = 0; j < TN; ++j) y[j] = in ? B[qb[j] + at * b_sk] : 0.0f;
                multiply_f32(x, y, 1);
            }
        }
        // acc[i][j][4g + r] holds C[row = 32i + 8g + 4*lh + r][col = 32j + li] of the wave's sub-tile
#pragma unroll
        for (int i = i0; i < i0 + ROWS; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int g = 0; g < 4; ++g)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const long long row = bm + wm * (32 * TM) + 32 * i + 8 * g + 4 * lh + r;
                    const long long col = bn + wn * (32 * TN) + 32 * j + li;
                    if (IN_RESULT(row, col))
                    {
                        const float sum_value = acc[i][j][4 * g + r] * unscale;
#if STORE_C
                        C[row * N + col] = sum_value;
#endif
                        EPILOGUE
                    }
                }
    }
}
)";
}

std::string gemm_split_kernel_source(const GemmConfig& cfg, const std::string& entry, const GemmEpilogue* epilogue) {
    std::string s = gemm_kernel_head(cfg, epilogue) + gemm_tile_head(cfg);
    const int per_thread = 8 * (int)gemm_threads(cfg);   // elements of an operand's tile that a thread's unit of eight k covers
    s += strf("#define BK %d\n#define KW %d\n#define PINGPONG %d\n#define KS %d\n#define RA_VALUE %d\n#define RB_VALUE %d\n", cfg.bk, cfg.k_waves,
              cfg.bm == 256 ? 1 : 0, cfg.bm == 256 ? cfg.bk / 16 : 1, cfg.bm * cfg.bk / per_thread, gemm_tile_columns(cfg) * cfg.bk / per_thread);
    s += R"(
#define KG (BK / 8)                     /* groups of eight k of a tile */
#define RA RA_VALUE                     /* rows of A (with their eight k) that a thread carries from memory to LDS */
#define RB RB_VALUE
#define LDA (BM + 4)                    /* rows of a k group in LDS: the next group starts a quarter of the banks on */
#define LDB (BN + 4)
#define WGN (BN / (32 * TN))            /* waves along n */
#define SCALE 65536.0f                  /* what the parts of an operand are larger by: its third part is then above bf16's smallest number */
#define SETS (KW == 1 && BK == 32 ? 2 : 1)   /* of accumulators: for the first and second half of a tile's k */
)" + split_types() + R"()" + gemm_entry(cfg, entry, epilogue, gemm_threads(cfg)) + R"(#if SPLITK
#if GROUPED
    const unsigned slice = blockIdx.z;  // c<y> points at problem y's own [gridDim.z][M][N] slices
#else
    const unsigned slice = blockIdx.y;
#endif
    const long long k_lo = (long long)slice * k_chunk;
    const long long k_hi = min(K, k_lo + k_chunk);
    C += (long long)slice * M * N;
#else
    const long long k_lo = 0, k_hi = K;
#endif
    __shared__ __attribute__((aligned(16))) uint4_t lds[2 * 3 * KG * (LDA + LDB)];
    uint4_t (*As)[3][KG][LDA] = (uint4_t (*)[3][KG][LDA])lds;
    uint4_t (*Bs)[3][KG][LDB] = (uint4_t (*)[3][KG][LDB])(lds + 2 * 3 * KG * LDA);

    const unsigned tid = threadIdx.x;
    const unsigned lane = tid & 63u, wave = tid >> 6;
    const unsigned wm = wave / WGN % (BM / (32 * TM)), wn = wave % WGN, kw = wave / (NT / 64 / KW);
    const unsigned li = lane & 31u, lh = lane >> 5;

    // Block -> tile, as in the kernel on the FP32 matrix cores: ids regrouped per XCD, then column-major groups of rows.
    const unsigned gm = (unsigned)((M + BM - 1) / BM), gn = (unsigned)((N + BN - 1) / BN);
    const unsigned nblk = gm * gn;
    unsigned pid = blockIdx.x;
    if ((nblk & 7u) == 0) pid = (pid & 7u) * (nblk >> 3) + (pid >> 3);
    const unsigned GROUP = 8;
    const unsigned per_group = GROUP * gn;
    const unsigned group = pid / per_group;
    const unsigned first_m = group * GROUP;
    const unsigned gsz = min(gm - first_m, GROUP);
    const unsigned tile_m = first_m + (pid % per_group) % gsz;
    const unsigned tile_n = (pid % per_group) / gsz;
    const long long bm = (long long)tile_m * BM, bn = (long long)tile_n * BN;

    A += a_off;
    B += b_off;

    float16_t sums[SETS][TM][TN];
    float16_t (&acc)[TM][TN] = sums[0];
#pragma unroll
    for (int s = 0; s < SETS; ++s)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) sums[s][i][j][r] = 0.0f;

    // What a thread carries of a k-tile: eight consecutive k of RA rows of A and of RB columns of B.  Along a
    // contiguous k its rows lie NT / KG apart and come as two 128-bit loads each; along contiguous rows they are
    // neighbours, loaded together for one k after the other.
#define ROW_A(i) (A_KCONTIG ? tid / KG + (NT / KG) * (i) : (tid % (BM / RA)) * RA + (i))
#define ROW_B(i) (B_KCONTIG ? tid / KG + (NT / KG) * (i) : (tid % (BN / RB)) * RB + (i))
    const unsigned ga = A_KCONTIG ? tid % KG : tid / (BM / RA), gb = B_KCONTIG ? tid % KG : tid / (BN / RB);
#if EDGE
    // rows beyond the product read its last row: what they contribute to is never stored
#define CLAMP_A(r) min(bm + (long long)(r), M - 1)
#define CLAMP_B(r) min(bn + (long long)(r), N - 1)
#define IN_RESULT(row, col) ((row) < M && (col) < N)
#else
#define CLAMP_A(r) (bm + (long long)(r))
#define CLAMP_B(r) (bn + (long long)(r))
#define IN_RESULT(row, col) true
#endif
    const int KT = __builtin_amdgcn_readfirstlane((int)((k_hi - k_lo + BK - 1) / BK));
#if EDGE
    // the last tile ends where k ends: if k is no multiple of the tile, it starts inside the tile before, and the first
    // `again` of its k, which that tile has had, are parked as zeros (K is at least BK)
    const int again = __builtin_amdgcn_readfirstlane((int)(KT * BK - (k_hi - k_lo)));
    const long long k_first = KT == 1 ? k_hi - BK : k_lo;
#else
    const long long k_first = k_lo;
#endif
#if EDGE
    const float *pa[RA], *pb[RB];
#pragma unroll
    for (int i = 0; i < RA; ++i) pa[i] = A + CLAMP_A(ROW_A(i)) * a_sm + (k_first + 8 * ga) * a_sk;
#pragma unroll
    for (int i = 0; i < RB; ++i) pb[i] = B + CLAMP_B(ROW_B(i)) * b_sn + (k_first + 8 * gb) * b_sk;
#define AT_A(i, q) (pa[i] + (q) * a_sk)
#define AT_B(i, q) (pb[i] + (q) * b_sk)
#else
    // a wave-uniform pointer, moved on by scalar instructions, and one 32-bit offset per thread and operand (the
    // caller keeps lines of 2^22 elements and more away)
    const float* pa = A + bm * a_sm + k_first * a_sk;
    const float* pb = B + bn * b_sn + k_first * b_sk;
    const unsigned oa = 4u * (ROW_A(0) * (unsigned)a_sm + 8u * ga * (unsigned)a_sk);
    const unsigned ob = 4u * (ROW_B(0) * (unsigned)b_sn + 8u * gb * (unsigned)b_sk);
#define AT_A(i, q) ((const float*)((const char*)(pa + (A_KCONTIG ? (i) * (long long)(NT / KG) * a_sm + (q) : (q) * a_sk + (i))) + oa))
#define AT_B(i, q) ((const float*)((const char*)(pb + (B_KCONTIG ? (i) * (long long)(NT / KG) * b_sn + (q) : (q) * b_sk + (i))) + ob))
#endif
    int t_at = 0;   // the tile that the next loads fetch; beyond the last one they fetch the last one again
    auto load_next = [&](float (*ra)[8], float (*rb)[8]) {
#if A_KCONTIG
#pragma unroll
        for (int i = 0; i < RA; ++i) {
            *(float4_t*)&ra[i][0] = *(const float4_g*)AT_A(i, 0);
            *(float4_t*)&ra[i][4] = *(const float4_g*)AT_A(i, 4);
        }
#else
#pragma unroll
        for (int q = 0; q < 8; ++q) {
#if EDGE || RA_VALUE == 1
#pragma unroll
            for (int i = 0; i < RA; ++i) ra[i][q] = *AT_A(i, q);
#else
#pragma unroll
            for (int i = 0; i < RA; i += 2) {
                const float2_t v = *(const float2_t*)AT_A(i, q);
                ra[i][q] = v.x;
                ra[i + 1][q] = v.y;
            }
#endif
        }
#endif
#if B_KCONTIG
#pragma unroll
        for (int i = 0; i < RB; ++i) {
            *(float4_t*)&rb[i][0] = *(const float4_g*)AT_B(i, 0);
            *(float4_t*)&rb[i][4] = *(const float4_g*)AT_B(i, 4);
        }
#else
#pragma unroll
        for (int q = 0; q < 8; ++q) {
#if EDGE || RB_VALUE == 1
#pragma unroll
            for (int i = 0; i < RB; ++i) rb[i][q] = *AT_B(i, q);
#else
#pragma unroll
            for (int i = 0; i < RB; i += 2) {
                const float2_t v = *(const float2_t*)AT_B(i, q);
                rb[i][q] = v.x;
                rb[i + 1][q] = v.y;
            }
#endif
        }
#endif
        const bool go = t_at + 1 < KT;
        int ahead = go ? BK : 0;
#if EDGE
        if (t_at + 2 == KT) ahead -= again;
#pragma unroll
        for (int i = 0; i < RA; ++i) pa[i] += ahead * a_sk;
#pragma unroll
        for (int i = 0; i < RB; ++i) pb[i] += ahead * b_sk;
#else
        pa += ahead * a_sk;
        pb += ahead * b_sk;
#endif
        t_at += go ? 1 : 0;
    };
    // The matrix cores align the products of a step with a loss that leans towards minus infinity, by some 5e-8 of a
    // sum's size over k = 1024: nothing beside the roundings, but of one sign everywhere, so that averages over many
    // results would show it.  Half of k is therefore summed up negated, A changing sign on its way to LDS: the
    // second half of each tile where it has accumulators of its own, else runs of tiles in the order + - - + - + + -
    // ..., which also cancels what grows with the sum; the accumulators change sign where a run ends.
#if KW == 2 || BK == 32
    const float a_scale = ga >= KG / 2 ? -SCALE : SCALE;
#define SCALE_OF(t) a_scale
#else
    const int run = 31 - __builtin_clz((unsigned)max(KT >> 3, 1));
    auto minus = [&](int t) { return (__builtin_popcount((unsigned)t >> run) & 1) != 0; };
#define SCALE_OF(t) (minus(t) ? -SCALE : SCALE)
    auto negate = [&] {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[i][j][r] = -acc[i][j][r];
    };
#endif
    auto park_one = [&](uint4_t* to, int plane, const float* r, float scale) {
        uint4_t p0, p1, p2;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            unsigned u0, u1, u2;
            split(r[2 * q], r[2 * q + 1], scale, u0, u1, u2);
            p0[q] = u0;
            p1[q] = u1;
            p2[q] = u2;
        }
        to[0] = p0;
        to[plane] = p1;
        to[2 * plane] = p2;
    };
    // tile t, which has been loaded, goes to LDS in parts
    auto park = [&](int buf, int t, const float (*ra)[8], const float (*rb)[8]) {
#pragma unroll
        for (int i = 0; i < RA; ++i) park_one(&As[buf][0][ga][ROW_A(i)], KG * LDA, ra[i], SCALE_OF(t));
#pragma unroll
        for (int i = 0; i < RB; ++i) park_one(&Bs[buf][0][gb][ROW_B(i)], KG * LDB, rb[i], SCALE);
    };
    // ... and if it is the last and has k that the tile before had, A is parked once more with zeros there.  (B keeps
    // its values: zero times what is finite is zero, and a sum that is not finite is computed again anyway.)
    auto park_rim = [&](int buf, int t, const float (*ra)[8]) {
#if EDGE
        if (t + 1 == KT && again > 0) {
#pragma unroll
            for (int i = 0; i < RA; ++i) {
                float r[8];
#pragma unroll
                for (int q = 0; q < 8; ++q) r[q] = (int)(8 * ga + q) < again ? 0.0f : ra[i][q];
                park_one(&As[buf][0][ga][ROW_A(i)], KG * LDA, r, SCALE_OF(t));
            }
        }
#endif
    };
    // One k-tile.  Of the nine products of parts the six that reach the result's 24 bits are taken, the smallest first.
    bf16x8_t fa[KS][3][TM], fb[KS][3][TN];
    auto read_parts = [&](int cur, int ks, int at) {
#pragma unroll
        for (int p = 0; p < 3; ++p) {
#pragma unroll
            for (int i = 0; i < TM; ++i) fa[at][p][i] = __builtin_bit_cast(bf16x8_t, As[cur][p][2 * ks + lh][wm * (32 * TM) + 32 * i + li]);
#pragma unroll
            for (int j = 0; j < TN; ++j) fb[at][p][j] = __builtin_bit_cast(bf16x8_t, Bs[cur][p][2 * ks + lh][wn * (32 * TN) + 32 * j + li]);
        }
    };
#define TERM(x, y)                                          \
            _Pragma("unroll") for (int i = 0; i < TM; ++i)  \
            _Pragma("unroll") for (int j = 0; j < TN; ++j)  \
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[at][x][i], fb[at][y][j], acc[i][j], 0, 0, 0);
    auto multiply = [&](int at, float16_t (&acc)[TM][TN]) {
        TERM(2, 0)
        TERM(0, 2)
        TERM(1, 1)
        TERM(1, 0)
        TERM(0, 1)
        TERM(0, 0)
    };

    float ra0[RA][8], rb0[RB][8];
#if PINGPONG
    // The two wavefronts of a SIMD take turns: while one multiplies, the other reads its next operands from LDS, splits
    // and parks the tile after that and asks memory for the one behind it.  The second four wavefronts run half a
    // tile behind the first: a barrier more at the start, one fewer at the end.
    auto meet = [&] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    };
    const bool second = __builtin_amdgcn_readfirstlane((int)wave) >= NT / 128;
    load_next(ra0, rb0);
    park(0, 0, ra0, rb0);
    park_rim(0, 0, ra0);
    load_next(ra0, rb0);
    meet();
    if (second) meet();
    for (int kt = 0; kt < KT; ++kt) {
        if (kt > 0 && minus(kt) != minus(kt - 1)) negate();
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) read_parts(kt & 1, ks, ks);
        park((kt & 1) ^ 1, kt + 1, ra0, rb0);
        park_rim((kt & 1) ^ 1, kt + 1, ra0);
        load_next(ra0, rb0);
        meet();
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) multiply(ks, acc);
        __builtin_amdgcn_s_setprio(0);
        meet();
    }
    if (!second) meet();
#else
    float ra1[RA][8], rb1[RB][8];
#if KW == 1 && BK == 16
#define NEGATE_AT(t) if ((t) > 0 && minus(t) != minus((t) - 1)) negate();
#else
#define NEGATE_AT(t)
#endif
    // the vector instructions that split the next tile go between the matrix instructions, which leave them room (a
    // wavefront with one block has a short chain of them, and does better when the compiler places them)
#if TM * TN > 1
#define MATRIX_OPS (6 * TM * TN * (BK / 16 / KW))   /* of a wavefront in a tile */
#define INTERLEAVE                                                                                          \
    _Pragma("unroll") for (int q = 0; q < MATRIX_OPS; ++q) {                                                \
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                                                  \
        __builtin_amdgcn_sched_group_barrier(0x002, (48 * RA + 48 * RB + MATRIX_OPS - 1) / (MATRIX_OPS) + 1, 0); \
    }
#else
#define INTERLEAVE
#endif
    auto compute = [&](int cur) {
#pragma unroll
        for (int ks = 0; ks < BK / 16 / KW; ++ks) {
            read_parts(cur, kw * (BK / 16 / KW) + ks, 0);
            multiply(0, sums[ks & (SETS - 1)]);
        }
    };
    load_next(ra0, rb0);
    load_next(ra1, rb1);
    park(0, 0, ra0, rb0);
    park_rim(0, 0, ra0);
    __syncthreads();
    int kt = 0;
    for (; kt + 1 < KT; kt += 2) {
        NEGATE_AT(kt)
        load_next(ra0, rb0);
        compute(0);
        park(1, kt + 1, ra1, rb1);
        INTERLEAVE
        park_rim(1, kt + 1, ra1);
        __syncthreads();
        NEGATE_AT(kt + 1)
        load_next(ra1, rb1);
        compute(1);
        park(0, kt + 2, ra0, rb0);
        INTERLEAVE
        park_rim(0, kt + 2, ra0);
        __syncthreads();
    }
    if (kt < KT) {
        NEGATE_AT(kt)
        compute(0);
    }
#endif
#if KW == 1 && BK == 16
    if (minus(KT - 1)) negate();
#elif KW == 1
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] -= sums[1][i][j];
#endif

#if KW == 2
    // the wavefronts that had the second half of every tile's k hand their sums to those that had the first
    {
        __syncthreads();
        float* mine = (float*)lds + (size_t)((wave % (NT / 128)) * 64 + lane) * 4;
        constexpr unsigned stride = NT / 128 * 64 * 4;
        if (kw == 1) {
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int g = 0; g < 4; ++g)
                        *(float4_t*)(mine + (4 * (i * TN + j) + g) * stride) =
                            float4_t{acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
        }
        __syncthreads();
        if (kw == 1) return;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const float4_t v = *(const float4_t*)(mine + (4 * (i * TN + j) + g) * stride);
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[i][j][4 * g + r] -= v[r];
                }
    }
#endif

)" + split_tail();
    return s;
}

}  // namespace adhip
