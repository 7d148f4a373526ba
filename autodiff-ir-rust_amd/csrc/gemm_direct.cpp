// FP32 matrix product for gfx950 on the bf16 matrix cores without a staging buffer: small outputs.
//
// The arithmetic is that of gemm_split.cpp (three bf16 parts an operand, six products of parts).  There a tile's operands
// are split once, stand in LDS and are read by every wavefront that needs them; between two barriers all wavefronts read LDS,
// then all multiply, then all split and write, and a k-tile of 64x64x64 took 0.93 us on a block's own CU where its matrix
// instructions take 0.32.  Here k is shared between the eight wavefronts of a block instead: each multiplies the whole
// tile by every eighth step of 32 k, with operands that go from memory to the registers the matrix instructions read.  No
// element is split twice for that (a step's k belong to one wavefront), there is no barrier before the end, and the splitting
// of the next half step stands between the matrix instructions of this one.  At the end the eight partial results are added
// through LDS in a fixed order.  Errors against 64 bits are half of one sum over k (k = 1000: 1.7e-7 for 3.4e-7).
//
// Tiles of 64x64, 64x32, 32x64 and 32x32; 8.2, 6.2 and 4.3 ns per k on a CU (64x64 staged through LDS: 14.5).  What bounds
// it is the issue of vector instructions: 13 for a pair of numbers, at five cycles each, leave the matrix cores busy 60 % of
// the time at 64x64.  Sixteen wavefronts for a 32x32 tile are no faster.  Whole launches, staged -> this: 1000 x 500 x 784
// 20.2 -> 15.2 us, 784 x 500 x 1000 24.1 -> 16.3, 500 x 320 x 1000 22.1 -> 12.0, 300 x 10 x 1000 22.4 -> 11.7 (of which 5.5 are
// the launch itself).
#include "gemm.hpp"

#include "common.hpp"

namespace adhip {

std::string gemm_direct_kernel_source(const GemmConfig& cfg, const std::string& entry, const GemmEpilogue* epilogue) {
    const int tm = cfg.bm / 32, tn = cfg.bn / 32;
    ADHIP_CHECK(cfg.k_waves == kDirectWaves && cfg.bk == 32 && (tm == 1 || tm == 2) && (tn == 1 || tn == 2), "internal: configuration of the kernels that stage through LDS");
    std::string s = gemm_kernel_head(cfg, epilogue);
    s += strf("#define RM %d\n#define RN %d\n#define TM 1\n#define TN 1\n#define WAVES %d\n#define A_NARROW %d\n#define B_NARROW %d\n#define OFFSET %s\n", tm, tn,
              cfg.k_waves, cfg.narrow_m ? 1 : 0, cfg.narrow_n ? 1 : 0, cfg.wide_lines ? "unsigned long long" : "unsigned");
    s += R"(
#define BM (32 * RM)
#define BN (32 * RN)
#define BK 32                           /* k of a step */
#define LD (BM + 4)                     /* a column of a partial result in LDS: four banks on from the one before */
#define SCALE 65536.0f                  /* what the parts of an operand are larger by: its third part is then above bf16's smallest number */
#define A_PAIRS (RM == 2 && !A_KCONTIG && !A_NARROW)   /* a lane's two rows of A are neighbours, and come as one 64-bit load */
#define B_PAIRS (RN == 2 && !B_KCONTIG && !B_NARROW)
#define LINES_A (A_KCONTIG ? BM * BK : 0)              /* a wavefront's floats of LDS for operands that go through it */
#define LINES_B (B_KCONTIG ? BN * BK : 0)
#define PART (BN * LD)                                 /* ... and for its partial result */
#define LDS_WAVE (LINES_A + LINES_B > PART ? LINES_A + LINES_B : PART)
)" + split_types() + gemm_entry(cfg, entry, epilogue, gemm_threads(cfg)) + R"(
    typedef float2_t float2_g UNALIGNED;
#if SPLITK
#if GROUPED
    const unsigned slice = blockIdx.z;
#else
    const unsigned slice = blockIdx.y;
#endif
    const long long k_lo = (long long)slice * k_chunk;
    const long long k_hi = min(K, k_lo + k_chunk);
    C += (long long)slice * M * N;
#else
    const long long k_lo = 0, k_hi = K;
#endif
    __shared__ __attribute__((aligned(16))) float lds[WAVES * LDS_WAVE];

    const unsigned lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const unsigned li = lane & 31u, lh = lane >> 5;

    // Block -> tile: ids regrouped per XCD, then column-major groups of rows, as in the kernels that stage through LDS.
    const unsigned gm = (unsigned)((M + BM - 1) / BM), gn = (unsigned)((N + BN - 1) / BN);
    const unsigned nblk = gm * gn;
    unsigned pid = blockIdx.x;
    if ((nblk & 7u) == 0) pid = (pid & 7u) * (nblk >> 3) + (pid >> 3);
    const unsigned GROUP = 8;
    const unsigned per_group = GROUP * gn;
    const unsigned group = pid / per_group;
    const unsigned first_m = group * GROUP;
    const unsigned gsz = min(gm - first_m, GROUP);
    const long long own_m = (long long)(first_m + (pid % per_group) % gsz) * BM, own_n = (long long)((pid % per_group) / gsz) * BN;
    // A tile that would reach beyond the product is moved back inside it (what it shares with the one before is not
    // stored), so that no load needs a condition; a product of fewer than 64 rows repeats its last one.
#if EDGE
    const long long bm = A_NARROW ? 0 : min(own_m, M - BM), bn = B_NARROW ? 0 : min(own_n, N - BN);
#define CLAMP_A(r) min(bm + (long long)(r), M - 1)
#define CLAMP_B(r) min(bn + (long long)(r), N - 1)
#define IN_RESULT(row, col) ((row) >= own_m && (row) < M && (col) >= own_n && (col) < N)
#else
    const long long bm = own_m, bn = own_n;
#define CLAMP_A(r) (bm + (long long)(r))
#define CLAMP_B(r) (bn + (long long)(r))
#define IN_RESULT(row, col) true
#endif
    A += a_off;
    B += b_off;

    // The last step ends where k ends, and the steps before it end where the next begins.  If k is no multiple of 32 the
    // first one begins where k does all the same, and those of its k that belong to the second are zeros of A (K is at
    // least 32; a range of fewer k begins its only step in front of itself, and what lies there is taken as zeros).
    const int steps = __builtin_amdgcn_readfirstlane((int)((k_hi - k_lo + BK - 1) / BK));
    const long long k_second = k_hi - (long long)(steps - 1) * BK;
    auto k_of_step = [&](int t) { return t > 0 || steps == 1 ? k_second + (long long)(t - 1) * BK : k_lo; };

    // What a lane multiplies of 16 k: eight k of two rows (i = 0, 1) of A and of two columns of B, the eight k being
    // 8 (q / 4) + 4 lh + q % 4.  Along contiguous rows these are the neighbours 2 li and 2 li + 1 of the tile and come
    // as one 64-bit load.  Along a contiguous k they are li and li + 32, and lanes side by side would read one line each, 16
    // bytes a cycle: such an operand is loaded eight lanes to a line of 32 k and goes through the wavefront's own 8 KB of LDS,
    // its 128-bit words in the order of their number times (exclusive or) the line's, which keeps reads and writes off one another's banks.
#define K_OF(q) (8 * ((q) >> 2) + 4 * (int)lh + ((q) & 3))
#define UNIFORM_K(q) (8 * ((q) >> 2) + ((q) & 3))
    const unsigned line_of = lane >> 3, word_of = lane & 7u;
    OFFSET oa[A_KCONTIG && A_NARROW ? 4 * RM : RM], ob[B_KCONTIG && B_NARROW ? 4 * RN : RN];   // bytes from the step's first element
#if A_KCONTIG
#pragma unroll
    for (int i = 0; i < (A_NARROW ? 4 * RM : 1); ++i) oa[i] = 4u * ((OFFSET)(A_NARROW ? min(8 * i + line_of, (unsigned)M - 1u) : line_of) * (OFFSET)a_sm + 4u * word_of);
#define AT_A(i) ((const char*)(pa + (A_NARROW ? 0 : 8 * (i)) * a_sm) + oa[A_NARROW ? (i) : 0])
#else
#pragma unroll
    for (int i = 0; i < RM; ++i) oa[i] = 4u * ((OFFSET)(A_NARROW ? min(RM * li + i, (unsigned)M - 1u) : RM * li) + 4u * lh * (OFFSET)a_sk);
#define AT_A(k, i) ((const char*)(pa + (k) * a_sk) + oa[i])
#endif
#if B_KCONTIG
#pragma unroll
    for (int i = 0; i < (B_NARROW ? 4 * RN : 1); ++i) ob[i] = 4u * ((OFFSET)(B_NARROW ? min(8 * i + line_of, (unsigned)N - 1u) : line_of) * (OFFSET)b_sn + 4u * word_of);
#define AT_B(i) ((const char*)(pb + (B_NARROW ? 0 : 8 * (i)) * b_sn) + ob[B_NARROW ? (i) : 0])
#else
#pragma unroll
    for (int i = 0; i < RN; ++i) ob[i] = 4u * ((OFFSET)(B_NARROW ? min(RN * li + i, (unsigned)N - 1u) : RN * li) + 4u * lh * (OFFSET)b_sk);
#define AT_B(k, i) ((const char*)(pb + (k) * b_sk) + ob[i])
#endif
    const float* from_a = A + bm * a_sm;
    const float* from_b = B + bn * b_sn;
    float ra[2][RM][8], rb[2][RN][8];   // the two halves of a step
#if A_KCONTIG
    float4_t ga[4 * RM];                   // a step on its way to LDS
    float4_t* const la = (float4_t*)lds + wave * LDS_WAVE / 4;
#endif
#if B_KCONTIG
    float4_t gb[4 * RN];
    float4_t* const lb = (float4_t*)lds + (wave * LDS_WAVE + LINES_A) / 4;
#endif
    // asks memory for the operands that go through LDS, a whole step, or for half a step of the others
    auto load_lines = [&](long long k) {
        const float* pa = from_a + k * a_sk;
        const float* pb = from_b + k * b_sk;
#if A_KCONTIG
#pragma unroll
        for (int i = 0; i < 4 * RM; ++i) ga[i] = *(const float4_g*)AT_A(i);
#endif
#if B_KCONTIG
#pragma unroll
        for (int i = 0; i < 4 * RN; ++i) gb[i] = *(const float4_g*)AT_B(i);
#endif
    };
    auto load_half = [&](long long k, int h) {
        const float* pa = from_a + (k + 16 * h) * a_sk;
        const float* pb = from_b + (k + 16 * h) * b_sk;
#if !A_KCONTIG
#pragma unroll
        for (int q = 0; q < 8; ++q) {
#if A_PAIRS
            const float2_t v = *(const float2_g*)AT_A(UNIFORM_K(q), 0);
            ra[h][0][q] = v.x;
            ra[h][RM - 1][q] = v.y;
#else
#pragma unroll
            for (int i = 0; i < RM; ++i) ra[h][i][q] = *(const float*)AT_A(UNIFORM_K(q), i);
#endif
        }
#endif
#if !B_KCONTIG
#pragma unroll
        for (int q = 0; q < 8; ++q) {
#if B_PAIRS
            const float2_t v = *(const float2_g*)AT_B(UNIFORM_K(q), 0);
            rb[h][0][q] = v.x;
            rb[h][RN - 1][q] = v.y;
#else
#pragma unroll
            for (int i = 0; i < RN; ++i) rb[h][i][q] = *(const float*)AT_B(UNIFORM_K(q), i);
#endif
        }
#endif
    };
    // (a wavefront's LDS accesses are carried out in order; the compiler only has to keep them in order too)
    auto in_order = [&] {
#if A_KCONTIG || B_KCONTIG
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#endif
    };
    auto park_lines = [&] {
        in_order();
#if A_KCONTIG
#pragma unroll
        for (int i = 0; i < 4 * RM; ++i) la[(8 * i + line_of) * 8 + (word_of ^ line_of)] = ga[i];
#endif
#if B_KCONTIG
#pragma unroll
        for (int i = 0; i < 4 * RN; ++i) lb[(8 * i + line_of) * 8 + (word_of ^ line_of)] = gb[i];
#endif
        in_order();
    };
    auto read_half = [&](int h) {
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const unsigned at = li * 8 + ((4 * h + 2 * c + lh) ^ (li & 7u));
#if A_KCONTIG
#pragma unroll
            for (int i = 0; i < RM; ++i) *(float4_t*)&ra[h][i][4 * c] = la[at + 256 * i];
#endif
#if B_KCONTIG
#pragma unroll
            for (int i = 0; i < RN; ++i) *(float4_t*)&rb[h][i][4 * c] = lb[at + 256 * i];
#endif
        }
    };

    float16_t part[RM][RN];
#pragma unroll
    for (int i = 0; i < RM; ++i)
#pragma unroll
        for (int j = 0; j < RN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) part[i][j][r] = 0.0f;
    // The matrix cores align the products of a step with a loss that leans towards minus infinity: half of the wavefronts
    // take A with the other sign, and their results are subtracted.
    const float a_scale = (__builtin_popcount(wave) & 1) ? -SCALE : SCALE;
    bf16x8_t fa[2][3][RM], fb[2][3][RN];   // half a step in parts
    // (part by part and not number by number: the parts of the half step before are used up in the opposite order)
    auto split_half = [&](int h) {
        uint4_t ua[3][RM], ub[3][RN];
#pragma unroll
        for (int p = 0; p < 3; ++p)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
#pragma unroll
                for (int i = 0; i < RM; ++i) ua[p][i][q] = split_part(p, ra[h][i][2 * q], ra[h][i][2 * q + 1], a_scale);
#pragma unroll
                for (int j = 0; j < RN; ++j) ub[p][j][q] = split_part(p, rb[h][j][2 * q], rb[h][j][2 * q + 1], SCALE);
            }
#pragma unroll
        for (int p = 0; p < 3; ++p) {
#pragma unroll
            for (int i = 0; i < RM; ++i) fa[h][p][i] = __builtin_bit_cast(bf16x8_t, ua[p][i]);
#pragma unroll
            for (int j = 0; j < RN; ++j) fb[h][p][j] = __builtin_bit_cast(bf16x8_t, ub[p][j]);
        }
    };
    // of the nine products of parts the six that reach the result's 24 bits, the smallest first
#define TERM(x, y)                                          \
            _Pragma("unroll") for (int i = 0; i < RM; ++i)  \
            _Pragma("unroll") for (int j = 0; j < RN; ++j)  \
                part[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[h][x][i], fb[h][y][j], part[i][j], 0, 0, 0);
    auto multiply = [&](int h) {
        TERM(2, 0)
        TERM(0, 2)
        TERM(1, 1)
        TERM(1, 0)
        TERM(0, 1)
        TERM(0, 0)
    };
    // between two matrix instructions the splitting of the next half step
#define INTERLEAVE                                                \
    _Pragma("unroll") for (int q = 0; q < 6 * RM * RN; ++q) {     \
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);        \
        __builtin_amdgcn_sched_group_barrier(0x002, (54 * (RM + RN) + 6 * RM * RN - 1) / (6 * RM * RN), 0); \
    }
    // A step's two halves: while one is multiplied, the next is split.  The first pass multiplies zeros, which keeps the code
    // in one copy: a wavefront makes one to four passes, and most of what it executes it executes for the first time.
#pragma unroll
    for (int p = 0; p < 3; ++p) {
#pragma unroll
        for (int i = 0; i < RM; ++i) fa[1][p][i] = __builtin_bit_cast(bf16x8_t, uint4_t{0u, 0u, 0u, 0u});
#pragma unroll
        for (int j = 0; j < RN; ++j) fb[1][p][j] = __builtin_bit_cast(bf16x8_t, uint4_t{0u, 0u, 0u, 0u});
    }
    if ((int)wave < steps) {
        const long long k = k_of_step((int)wave);
        load_lines(k);
        load_half(k, 0);
        load_half(k, 1);
#if EDGE
        if (wave == 0 && (k < k_lo || k + BK > k_second)) {
            const int lo = (int)(k_lo - k), hi = (int)((steps == 1 ? k_hi : k_second) - k);
#if A_KCONTIG
#pragma unroll
            for (int i = 0; i < 4 * RM; ++i)
#pragma unroll
                for (int q = 0; q < 4; ++q) ga[i][q] = 4 * (int)word_of + q >= lo && 4 * (int)word_of + q < hi ? ga[i][q] : 0.0f;
#else
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int i = 0; i < RM; ++i)
#pragma unroll
                    for (int q = 0; q < 8; ++q) ra[h][i][q] = 16 * h + K_OF(q) >= lo && 16 * h + K_OF(q) < hi ? ra[h][i][q] : 0.0f;
#endif
        }
#endif
    }
#pragma unroll 1
    for (int t = (int)wave; t < steps; t += WAVES) {
        const long long k = k_of_step(t + WAVES < steps ? t + WAVES : t);   // (behind its last step a wavefront fetches that once more)
        park_lines();
        load_lines(k);
        read_half(0);
        __builtin_amdgcn_sched_barrier(0);
        multiply(1);
        split_half(0);
        INTERLEAVE
        read_half(1);
        load_half(k, 0);
        __builtin_amdgcn_sched_barrier(0);
        multiply(0);
        split_half(1);
        INTERLEAVE
        load_half(k, 1);
    }
    if ((int)wave < steps) multiply(1);
#if A_KCONTIG || B_KCONTIG
    __syncthreads();   // (a wavefront's partial result takes the place of its own lines, which it has read by then)
#endif
    // Partial results go to LDS column by column (part[i][j][4 g + r] is row 8 g + 4 lh + r of block i, column li of
    // block j), and a wavefront for each 32x32 block adds them up.
    if ((int)wave < steps) {
        float* mine = lds + wave * LDS_WAVE;
#pragma unroll
        for (int j = 0; j < RN; ++j) {
            float* column = mine + (B_KCONTIG ? li + 32 * j : RN * li + j) * LD;
#pragma unroll
            for (int g = 0; g < 4; ++g) {
#if A_KCONTIG || RM == 1
#pragma unroll
                for (int i = 0; i < RM; ++i) {
                    const float16_t& x = part[i][j];
                    *(float4_t*)(column + 32 * i + 8 * g + 4 * lh) = float4_t{x[4 * g], x[4 * g + 1], x[4 * g + 2], x[4 * g + 3]};
                }
#else
                const float16_t &x = part[0][j], &y = part[1][j];
                *(float4_t*)(column + 16 * g + 8 * lh) = float4_t{x[4 * g], y[4 * g], x[4 * g + 1], y[4 * g + 1]};
                *(float4_t*)(column + 16 * g + 8 * lh + 4) = float4_t{x[4 * g + 2], y[4 * g + 2], x[4 * g + 3], y[4 * g + 3]};
#endif
            }
        }
    }
    __syncthreads();
    if (wave >= RM * RN) return;
    const unsigned wm = wave / RN, wn = wave % RN;
    float16_t acc[1][1];
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[0][0][r] = 0.0f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
        if (w < steps) {
            const float* theirs = lds + w * LDS_WAVE + (32 * wn + li) * LD + 32 * wm + 4 * lh;
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const float4_t v = *(const float4_t*)(theirs + 8 * g);
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[0][0][4 * g + r] += (__builtin_popcount(w) & 1) ? -v[r] : v[r];
            }
        }
    }

)" + split_tail();
    return s;
}

}  // namespace adhip
