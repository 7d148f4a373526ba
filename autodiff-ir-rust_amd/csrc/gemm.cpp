// FP32 matrix product for gfx950 on the FP32 matrix cores (v_mfma_f32_32x32x2_f32), LDS-tiled: the kernel of products
// whose k is shorter than 32.  Longer ones run on the bf16 matrix cores (gemm_split.cpp), which share its interface.
//
// The reference multiplies with one work-item per output element, a sequential k loop and two
// global loads per multiply-add (reference src/devices/opencl/kernels/dotprod.rs:23-53); transposed
// operands are folded into its index expressions.  Here both operands are described by strides
// (so x^T and W^T of the backward pass need no copy), staged through LDS in 256x128x16, 128x128x16 or
// 64x64x16 tiles with the global loads two tiles ahead in registers.  A wavefront owns a 64x64 sub-tile (2x2 MFMA
// blocks of 32x32) in the two large tiles and one 32x32 block in the small one, which exists so that
// products with a small output still put a few hundred blocks on the chip.
#include "gemm.hpp"

#include <algorithm>
#include <cstdlib>

#include "common.hpp"

namespace adhip {

int gemm_tile_columns(const GemmConfig& cfg) { return cfg.bn ? cfg.bn : (cfg.bm == 64 ? 64 : 128); }

// 32x32 blocks of a wavefront's sub-tile, in rows and columns
static int wave_rows(const GemmConfig& cfg) { return cfg.bm == 256 && cfg.bf16_parts ? 4 : cfg.bm == 64 ? 1 : 2; }
static int wave_columns(const GemmConfig& cfg) { return gemm_tile_columns(cfg) == 64 ? 1 : 2; }
unsigned gemm_threads(const GemmConfig& cfg) {
    if (cfg.k_waves == kDirectWaves) return 64u * (unsigned)cfg.k_waves;
    return 64u * (unsigned)((cfg.bm / (32 * wave_rows(cfg))) * (gemm_tile_columns(cfg) / (32 * wave_columns(cfg))) * cfg.k_waves);
}

size_t gemm_lds_bytes(const GemmConfig& cfg) {
    const size_t bm = (size_t)cfg.bm, bn = (size_t)gemm_tile_columns(cfg), bk = (size_t)cfg.bk;
    if (!cfg.bf16_parts) return 4 * 2 * bk * (bm + 4 + bn + 4);
    if (cfg.k_waves != kDirectWaves) return 16 * 2 * 3 * (bk / 8) * (bm + 4 + bn + 4);
    const size_t lines = (cfg.a_kcontig ? bm * bk : 0) + (cfg.b_kcontig ? bn * bk : 0);
    return 4 * kDirectWaves * std::max(lines, bn * (bm + 4));
}

std::string gemm_kernel_head(const GemmConfig& cfg, const GemmEpilogue* epilogue) {
    std::string s;
    if (epilogue) s += epilogue->prelude;
    s += strf("#define STORE_C %d\n", (!epilogue || epilogue->store_c) ? 1 : 0);
    {
        // the epilogue statements become one macro (line continuations), expanded where an element is finished
        std::string body = epilogue ? epilogue->code : std::string();
        std::string m = "#define EPILOGUE";
        size_t pos = 0;
        while (pos < body.size()) {
            size_t nl = body.find('\n', pos);
            if (nl == std::string::npos) nl = body.size();
            m += " \\\n    " + body.substr(pos, nl - pos);
            pos = nl + 1;
        }
        s += m + "\n";
    }
    s += strf("#define A_KCONTIG %d\n#define B_KCONTIG %d\n#define EDGE %d\n#define EDGE_VEC %d\n#define SPLITK %d\n#define GROUPED %d\n", cfg.a_kcontig ? 1 : 0,
              cfg.b_kcontig ? 1 : 0, cfg.edge ? 1 : 0, cfg.edge && cfg.edge_vec ? 1 : 0, cfg.split_k ? 1 : 0, cfg.grouped ? 1 : 0);
    return s;
}

std::string gemm_tile_head(const GemmConfig& cfg) {
    return strf("#define BM %d\n#define BN %d\n#define TM %d\n#define TN %d\n#define NT %u\n", cfg.bm, gemm_tile_columns(cfg), wave_rows(cfg),
                wave_columns(cfg), gemm_threads(cfg));
}

std::string gemm_entry(const GemmConfig& cfg, const std::string& entry, const GemmEpilogue* epilogue, unsigned threads, const char* more) {
    std::string s = strf("extern \"C\" __global__ __launch_bounds__(%u) void %s(const int* __restrict__ guard, ", threads, entry.c_str());
    const char* sizes = "long long M, long long N, long long K, ";
    if (cfg.grouped) {
        // one parameter triple per problem slot, and the (wave-uniform) choice among them by blockIdx.y
        std::string pick;
        for (int i = 0; i < kGemmGroupSlots; ++i) {
            s += strf("float* c%d, const float* a%d, const float* b%d, ", i, i, i);
            pick += strf("    case %d: C = c%d; A = a%d; B = b%d; break;\n", i, i, i, i);
        }
        return s + sizes + "long long a_sm, long long a_sk, long long b_sk, long long b_sn" + (cfg.split_k ? ", long long k_chunk" : "") + more + R"() {
    if (guard && *guard == 0) return;
    float* __restrict__ C;
    const float* __restrict__ A;
    const float* __restrict__ B;
    switch (blockIdx.y) {
)" + pick + "    default: return;\n    }\n    const long long a_off = 0, b_off = 0;\n";
    }
    return s + "float* __restrict__ C, const float* __restrict__ A, const float* __restrict__ B, " + sizes +
           "long long a_off, long long a_sm, long long a_sk, long long b_off, long long b_sk, long long b_sn" + (cfg.split_k ? ", long long k_chunk" : "") + more +
           (epilogue ? epilogue->params : std::string()) + ") {\n    if (guard && *guard == 0) return;\n";
}

std::string gemm_kernel_source(const GemmConfig& cfg, const std::string& entry, const GemmEpilogue* epilogue) {
    ADHIP_CHECK(!cfg.bf16_parts && !cfg.split_k && cfg.bk == 16 && cfg.k_waves == 1, "internal: configuration of the kernel on the bf16 matrix cores");
    std::string s = gemm_kernel_head(cfg, epilogue);
    // tile geometry: BM x BN block tile, TM x TN MFMA blocks per wave, WGN waves along n
    s += gemm_tile_head(cfg);
    {
        // diagnostic: ADHIP_GEMM_AHEAD=1 keeps the global loads one k-tile ahead of the MFMAs instead of two
        int ahead = 2;
        if (const char* e = getenv("ADHIP_GEMM_AHEAD")) ahead = atoi(e) == 1 ? 1 : 2;
        s += strf("#define AHEAD %d\n", ahead);
    }
    s += R"(
#define BK 16
// An MFMA operand read from LDS.  Volatile and explicitly in the LDS address space: the compiler then issues one
// ds_read_b32 per operand with the whole tile offset in the instruction's 16-bit immediate field, instead of pairing
// neighbouring reads into ds_read2_b32, whose 8-bit offsets do not reach the next k-row, so that every pair needed a
// vector add for its base.  Vector ALU instructions and FP32 MFMAs do not overlap on a SIMD; the 14 adds per k-tile
// this removes are worth 2 % (4096^3: 0.827 -> 0.844 of the FP32 matrix peak).
#define LDS_OPERAND(x) (*(const volatile __attribute__((address_space(3))) float*)&(x))
#define LDA (BM + 4)
#define LDB (BN + 4)
#define WGN (BN / (32 * TN))            /* waves along n */
#define A_LOADS (BM * BK / 4 / NT)      /* float4 loads of the A tile per thread */
#define B_LOADS (BN * BK / 4 / NT)      /* float4 loads of the B tile per thread */
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef float float16_t __attribute__((ext_vector_type(16)));
// 128 bits of an operand that is only known to be 4-byte aligned (an odd leading dim or offset): still one
// global_load_dwordx4, which the hardware splits where it crosses a cache line
typedef float4_t float4_ua __attribute__((aligned(4)));

#if EDGE
// Four operand elements p[off + j * step], j = 0..3, of which the first `valid` (any integer; <= 0: none) exist; the
// others read as 0.  `step` is the operand's unit stride (the four run along its contiguous dim).  With EDGE_VEC
// (the operands' contiguous extents are at least 4) a thread whose
// four elements all exist takes them with one 128-bit load, as the kernel without EDGE does, and only the threads on
// the ragged rim fall back to single elements.  The common load sits under no condition (a thread of the rim reads
// the operand's first elements there, and an element that does not exist is read at the first element and replaced),
// so that the loads of a tile are in flight together.  With EDGE_VEC the kernel calls this only for the last,
// ragged k-tile and for quads that straddle the end of M or N: everywhere else a row or column beyond the product
// is replaced by one inside it (what it contributes to is never stored) and the load is the plain 128-bit one.
static __device__ __forceinline__ float4_t edge_load4(const float* p, long long off, long long step, long long valid) {
    float4_t v;
#if EDGE_VEC
    const bool whole = valid >= 4;
    v = *(const float4_ua*)(p + (whole ? off : 0));
    if (!whole)
#endif
    {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const bool ok = j < valid;
            const float x = p[ok ? off + j * step : 0];
            v[j] = ok ? x : 0.0f;
        }
    }
    return v;
}
#endif

// A is [M,K] with element strides (a_sm, a_sk); B is [K,N] with (b_sk, b_sn); C dense [M,N].
// A_KCONTIG: a_sk == 1 (else a_sm == 1).  B_KCONTIG: b_sk == 1 (else b_sn == 1).
// EDGE: M, N or K is not a multiple of the tile, or an operand is not 16-byte aligned.  Stores are bounds-checked;
// loads go through edge_load4 where an element may not exist (all of them without EDGE_VEC; with it, only the last
// ragged k-tile and quads that straddle the end of M or N).
// GROUPED: several independent products of one shape and one set of strides in a single launch; the block row
// blockIdx.y works on problem y, whose three base pointers (operand offsets already applied) are parameters
// c<y>, a<y>, b<y>.  For the same kind of product when there are many of them (the per-head projections of
// multi-head attention).
)" + gemm_entry(cfg, entry, epilogue, gemm_threads(cfg)) + R"(    const long long k_lo = 0, k_hi = K;
    __shared__ __attribute__((aligned(16))) float As[2][BK][LDA];
    __shared__ __attribute__((aligned(16))) float Bs[2][BK][LDB];

    const unsigned tid = threadIdx.x;
    const unsigned lane = tid & 63u, wave = tid >> 6;
    const unsigned wm = wave / WGN, wn = wave % WGN;
    const unsigned li = lane & 31u, lh = lane >> 5;

    // Block -> tile.  Consecutive block ids go to different XCDs (8 of them, each with its own L2), so
    // ids are first regrouped per XCD and then walked in column-major groups of 8 tile rows, which
    // keeps the A and B panels one XCD works on small.
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

    float16_t acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

    float4_t ra0[A_LOADS], rb0[B_LOADS];

    auto load_a = [&](long long k0, float4_t* ra) {
#pragma unroll
        for (int i = 0; i < A_LOADS; ++i) {
#if A_KCONTIG
            const unsigned kq = tid & 3u, mr = (tid >> 2) + (NT / 4) * i;
            const long long m = bm + mr, k = k0 + 4 * kq;
#if EDGE
            // rows beyond M only feed rows of the product that are never stored: they read the last row instead
            if (EDGE_VEC && k0 + BK <= k_hi) ra[i] = *(const float4_ua*)(A + min(m, M - 1) * a_sm + k);
            else ra[i] = edge_load4(A, m * a_sm + k * a_sk, a_sk, m < M ? k_hi - k : 0);
#else
            ra[i] = *(const float4_t*)(A + m * a_sm + k);
#endif
#else
            const unsigned mq = tid % (BM / 4), kr = tid / (BM / 4) + (NT / (BM / 4)) * i;
            const long long m = bm + 4 * mq, k = k0 + kr;
#if EDGE
            // a quad of rows that lies wholly beyond M reads the last whole quad instead; one that straddles M is
            // taken element by element
            if (EDGE_VEC && k0 + BK <= k_hi && (m + 4 <= M || m >= M)) ra[i] = *(const float4_ua*)(A + k * a_sk + min(m, (M - 4) & ~3ll));
            else ra[i] = edge_load4(A, m * a_sm + k * a_sk, a_sm, k < k_hi ? M - m : 0);
#else
            ra[i] = *(const float4_t*)(A + k * a_sk + m);
#endif
#endif
        }
    };
    auto load_b = [&](long long k0, float4_t* rb) {
#pragma unroll
        for (int i = 0; i < B_LOADS; ++i) {
#if B_KCONTIG
            const unsigned kq = tid & 3u, nr = (tid >> 2) + (NT / 4) * i;
            const long long n = bn + nr, k = k0 + 4 * kq;
#if EDGE
            if (EDGE_VEC && k0 + BK <= k_hi) rb[i] = *(const float4_ua*)(B + min(n, N - 1) * b_sn + k);
            else rb[i] = edge_load4(B, k * b_sk + n * b_sn, b_sk, n < N ? k_hi - k : 0);
#else
            rb[i] = *(const float4_t*)(B + n * b_sn + k);
#endif
#else
            const unsigned nq = tid % (BN / 4), kr = tid / (BN / 4) + (NT / (BN / 4)) * i;
            const long long n = bn + 4 * nq, k = k0 + kr;
#if EDGE
            if (EDGE_VEC && k0 + BK <= k_hi && (n + 4 <= N || n >= N)) rb[i] = *(const float4_ua*)(B + k * b_sk + min(n, (N - 4) & ~3ll));
            else rb[i] = edge_load4(B, k * b_sk + n * b_sn, b_sn, k < k_hi ? N - n : 0);
#else
            rb[i] = *(const float4_t*)(B + k * b_sk + n);
#endif
#endif
        }
    };
    auto store_tiles = [&](int buf, const float4_t* ra, const float4_t* rb) {
#pragma unroll
        for (int i = 0; i < A_LOADS; ++i) {
#if A_KCONTIG
            const unsigned kq = tid & 3u, mr = (tid >> 2) + (NT / 4) * i;
#pragma unroll
            for (int j = 0; j < 4; ++j) As[buf][4 * kq + j][mr] = ra[i][j];
#else
            const unsigned mq = tid % (BM / 4), kr = tid / (BM / 4) + (NT / (BM / 4)) * i;
            *(float4_t*)&As[buf][kr][4 * mq] = ra[i];
#endif
        }
#pragma unroll
        for (int i = 0; i < B_LOADS; ++i) {
#if B_KCONTIG
            const unsigned kq = tid & 3u, nr = (tid >> 2) + (NT / 4) * i;
#pragma unroll
            for (int j = 0; j < 4; ++j) Bs[buf][4 * kq + j][nr] = rb[i][j];
#else
            const unsigned nq = tid % (BN / 4), kr = tid / (BN / 4) + (NT / (BN / 4)) * i;
            *(float4_t*)&Bs[buf][kr][4 * nq] = rb[i];
#endif
        }
    };

    // One k-tile: 8 MFMA steps from LDS buffer `cur`; the operands of step ks+1 are fetched from LDS before the
    // four MFMAs of step ks are issued, and half way through the tile that was prefetched into registers (sa, sb)
    // is parked in the other LDS buffer, which nobody reads during this iteration.
    auto compute = [&](int cur, bool park, const float4_t* sa, const float4_t* sb) {
        float fa[TM][2], fb[TN][2];
#pragma unroll
        for (int i = 0; i < TM; ++i) fa[i][0] = LDS_OPERAND(As[cur][lh][wm * (32 * TM) + 32 * i + li]);
#pragma unroll
        for (int j = 0; j < TN; ++j) fb[j][0] = LDS_OPERAND(Bs[cur][lh][wn * (32 * TN) + 32 * j + li]);
#pragma unroll
        for (int ks = 0; ks < BK / 2; ++ks) {
            const int c = ks & 1, nx = c ^ 1;
            if (ks + 1 < BK / 2) {
#pragma unroll
                for (int i = 0; i < TM; ++i) fa[i][nx] = LDS_OPERAND(As[cur][2 * (ks + 1) + lh][wm * (32 * TM) + 32 * i + li]);
#pragma unroll
                for (int j = 0; j < TN; ++j) fb[j][nx] = LDS_OPERAND(Bs[cur][2 * (ks + 1) + lh][wn * (32 * TN) + 32 * j + li]);
            }
            __builtin_amdgcn_sched_barrier(0);  // keep the LDS reads ahead of the MFMAs that hide their latency
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[i][c], fb[j][c], acc[i][j], 0, 0, 0);
            if (ks == BK / 4 - 1 && park) store_tiles(cur ^ 1, sa, sb);
        }
    };

    const int KT = __builtin_amdgcn_readfirstlane((int)((k_hi - k_lo + BK - 1) / BK));   // (uniform: kept in a scalar register)
#if AHEAD == 2
    // Global loads run two k-tiles ahead of the MFMAs, in two register sets that take turns: during tile kt the loads
    // of tile kt + 2 are issued into the set that held tile kt (parked in LDS during tile kt - 1), and the set that
    // holds tile kt + 1, issued a whole tile earlier, is parked.  A load then has a k-tile and a half of MFMAs to
    // arrive instead of half a tile (which is some 500 cycles where a wavefront owns 64x32, less than a trip to
    // memory).  Measured when products of any k ran here, of which there are one or two tiles left: 4096 x 1024 x 4096 in
    // 276 / 268 / 251 us instead of 289 / 274 / 257.  The loop is unrolled by two so that the sets and the LDS buffers are
    // named, not indexed.
    // Loads and parkings stand under no condition: beyond the last tile the loads fetch the last tile again and the
    // parking writes a tile nobody reads.  (Under a condition, the wait in front of a parking also waits for the
    // newest loads, or the compiler moves the loads down to the parking that consumes them.)
    int t_at = 0;   // the tile the next loads fetch
#if EDGE
    auto load_next = [&](float4_t* ra, float4_t* rb) {
        load_a(k_lo + (long long)t_at * BK, ra);
        load_b(k_lo + (long long)t_at * BK, rb);
        t_at += t_at + 1 < KT ? 1 : 0;
    };
#else
    // Without bounds checks an address is a wave-uniform pointer -- the tile's corner, moved on from tile to tile and
    // from one of a thread's loads to its next by scalar instructions -- plus one 32-bit offset per thread and
    // operand that never changes: no vector instruction per load (vector instructions are paid in matrix time).
    const unsigned oa = A_KCONTIG ? (tid >> 2) * (unsigned)a_sm + 4u * (tid & 3u) : (tid / (BM / 4)) * (unsigned)a_sk + 4u * (tid % (BM / 4));
    const unsigned ob = B_KCONTIG ? (tid >> 2) * (unsigned)b_sn + 4u * (tid & 3u) : (tid / (BN / 4)) * (unsigned)b_sk + 4u * (tid % (BN / 4));
    const float* Ab = A + (A_KCONTIG ? bm * a_sm + k_lo : k_lo * a_sk + bm);
    const float* Bb = B + (B_KCONTIG ? bn * b_sn + k_lo : k_lo * b_sk + bn);
    const long long ia = A_KCONTIG ? (NT / 4) * a_sm : (NT / (BM / 4)) * a_sk;   // from one of a thread's loads to its next
    const long long ib = B_KCONTIG ? (NT / 4) * b_sn : (NT / (BN / 4)) * b_sk;
    const long long step_a = A_KCONTIG ? BK : BK * a_sk, step_b = B_KCONTIG ? BK : BK * b_sk;
    auto load_next = [&](float4_t* ra, float4_t* rb) {
#pragma unroll
        for (int i = 0; i < A_LOADS; ++i) ra[i] = *(const float4_t*)((const char*)(Ab + i * ia) + (size_t)(4u * oa));
#pragma unroll
        for (int i = 0; i < B_LOADS; ++i) rb[i] = *(const float4_t*)((const char*)(Bb + i * ib) + (size_t)(4u * ob));
        const bool go = t_at + 1 < KT;
        Ab += go ? step_a : 0;
        Bb += go ? step_b : 0;
        t_at += go ? 1 : 0;
    };
#endif
    float4_t ra1[A_LOADS], rb1[B_LOADS];
    load_next(ra0, rb0);
    store_tiles(0, ra0, rb0);
    load_next(ra1, rb1);
    __syncthreads();
    int kt = 0;
    for (; kt + 1 < KT; kt += 2) {
        load_next(ra0, rb0);
        compute(0, true, ra1, rb1);
        __syncthreads();
        load_next(ra1, rb1);
        compute(1, true, ra0, rb0);
        __syncthreads();
    }
    if (kt < KT) compute(0, false, ra1, rb1);   // an odd number of tiles: the last one sits in buffer 0
#else
    // The next tile's global loads are issued before the current tile is multiplied (one tile ahead).
    load_a(k_lo, ra0);
    load_b(k_lo, rb0);
    store_tiles(0, ra0, rb0);
    __syncthreads();

    for (long long kt = 0; kt < KT; ++kt) {
        const bool more = kt + 1 < KT;
        if (more) {
            load_a(k_lo + (kt + 1) * BK, ra0);
            load_b(k_lo + (kt + 1) * BK, rb0);
        }
        compute((int)(kt & 1), more, ra0, rb0);
        __syncthreads();
    }
#endif

    // acc[i][j][4g + r] holds C[row = 32i + 8g + 4*lh + r][col = 32j + li] of the wave's sub-tile
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int g = 0; g < 4; ++g)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const long long row = bm + wm * (32 * TM) + 32 * i + 8 * g + 4 * lh + r;
                    const long long col = bn + wn * (32 * TN) + 32 * j + li;
#if EDGE
                    if (row < M && col < N)
#endif
                    {
                        const float sum_value = acc[i][j][4 * g + r];
#if STORE_C
                        C[row * N + col] = sum_value;
#endif
                        EPILOGUE
                    }
                }
}
)";
    return s;
}

// Products too small for a matrix-core tile, and operands without a unit stride.  Bound by latency: a thread that walks
// k alone makes k dependent trips through two loads (64 x 48 x 64: 12 us, where an empty kernel takes 4).  `lanes` lanes
// (a power of two, at most 64) share a result instead, each with every lanes-th k, four of which are in flight at once;
// the caller picks lanes so that one round of four covers k where it can.
std::string dot_small_source(const std::string& entry, const GemmEpilogue* epilogue, bool grouped) {
    GemmConfig cfg;
    cfg.grouped = grouped;
    std::string s = gemm_kernel_head(cfg, epilogue);
    s += gemm_entry(cfg, entry, epilogue, 256, ", int lanes");
    s += R"(
    const unsigned share = threadIdx.x & (unsigned)(lanes - 1), per_block = 256u / (unsigned)lanes;
    const long long total = M * N, g = (long long)blockIdx.x * per_block + threadIdx.x / (unsigned)lanes;
    if (g < total) {
        const long long row = total <= 0x7fffffff ? (long long)((unsigned)g / (unsigned)N) : g / N, col = g - row * N;
        const float* pa = A + a_off + row * a_sm;
        const float* pb = B + b_off + col * b_sn;
        float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        for (long long k0 = share; k0 < K; k0 += 4 * lanes) {
            float x[4], y[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                // what lies beyond k is read at the first place and taken as 0
                const long long k = k0 + u * lanes;
                const bool ok = k < K;
                x[u] = pa[ok ? k * a_sk : 0];
                y[u] = pb[ok ? k * b_sk : 0];
                x[u] = ok ? x[u] : 0.0f;
                y[u] = ok ? y[u] : 0.0f;
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) acc[u] = __builtin_fmaf(x[u], y[u], acc[u]);
        }
        float sum_value = (acc[0] + acc[1]) + (acc[2] + acc[3]);
        for (int d = lanes >> 1; d > 0; d >>= 1) sum_value += __shfl_xor(sum_value, d);
        if (share == 0) {
#if STORE_C
            C[g] = sum_value;
#endif
            EPILOGUE
        }
    }
}
#undef EPILOGUE
#undef STORE_C
#undef A_KCONTIG
#undef B_KCONTIG
#undef EDGE
#undef EDGE_VEC
#undef SPLITK
#undef GROUPED
)";
    return s;
}

}  // namespace adhip
