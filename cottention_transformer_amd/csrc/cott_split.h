// fp32 storage on the bf16 matrix cores: every fp32 operand is split into T bf16 numbers and every product of the chunk
// recurrence
//     out_c = ((A_c B_c^T) o mask) C_c + A_c S_c ;   S_{c+1} = S_c + B_c^T C_c          (chunks of 32 positions)
// is formed from the products of those terms, accumulating in fp32.
//   T = 2 (padded head dims 64 x 64): x = hi + lo with 16 of the 24 significant bits, a b from three matrix instructions,
//     rel-L2 of o, dQ, dK, dV against fp64 6.3e-6.
//   T = 3 (128-wide heads): x = hi + mid + lo holds all 24 bits; the six products down to 2^-16 of a b.  What is left out, mid lo
//     + lo mid, is of either sign and at most 2^-24 of a product of two operands, 1.5 2^-23 of one with the state or a score
//     (SplitMode).  Rel-L2 against fp64 7.0e-8 .. 2.1e-7, where the fp32 matrix pipe, which these widths took before, gives
//     1.9e-7 .. 3.7e-7 and terms that are all cut 1.2e-7 .. 2.3e-7 (N63 .. N8192, D 80 .. 128, forward and gradients); every
//     entry 1.0078, the worst of cut terms, N1 .. N128: at most 4.7e-8, 1.2e-7 and 4.8e-7.  Rounding costs 1 to 3 % of the
//     times below.  A product within 2^-8 of the largest fp32 number may come out infinite.  The fp32 pipe is sixteen times
//     slower than the bf16 one.
// Structure: that of colscan_kernel (cott_colscan.h).
//   * Four compute wavefronts each own a quarter of the state's columns, all rows, in fp32 accumulators whose row order makes
//     them the operand of A_c S_c once they are split; they produce those columns of the output.
//   * Four loader wavefronts move fp32 rows global -> registers -> T tiles per operand in LDS, two chunks ahead, and form
//     the three live 16 x 16 score tiles once per workgroup.
//   * One barrier per chunk: the product of the scores with C_c is finished at the start of the next chunk.
// Why 32 positions: T = 3 at 128 x 128 fills LDS (156 KiB with both buffers); at T = 2 it takes 68 KiB and two workgroups fit
// a CU, a third of the score products falls away, and the state is packed twice as often.  The group sums run the same code
// without A, scores and outputs (SUMS).
// What bounds it: the vector instructions of the splits, which share the issue port with the matrix ones.  Per chunk and
// SIMD at T = 3, 128 x 128: matrix pipe 3744 cycles, splits (11 instructions per pair of numbers) 750 instructions; 7400
// cycles in all.  Splitting with the packed dot product (one instruction per difference instead of two) is slower: it waits
// for the matrix pipe.
// Measured (us, forward / gradients, back to back; before: T = 3 on the fp32 matrix pipe, T = 2 in chunks of 64 positions with
// one workgroup per CU):
//   1 x 16 x 2048 x 128    73 / 168 -> 48 / 79       8 x 16 x 1024 x 128   175 / 418 -> 97 / 219
//   1 x 4 x 8192 x 128     80 / 171 -> 51 / 83       2 x 16 x 1024 x 128 / 64   42 / 102 -> 31 / 74
//   1 x 16 x 63 x 128      20 / 20 -> 11 / 11        8 x 16 x 2048 x 64 (T = 2)   67 / 160 -> 63 / 132
//   1 x 16 x 4096 x 64 (T = 2)   33 / 57 -> 27 / 43
// dV's state is the transpose of dK's where the padded dims are square: the sums are formed once and dV's scan reads them
// transposed, four dwords a tile and lane (gradients of 16 heads N2048 D128 96 -> 88 us, 8 heads N4096 94.5 -> 90, 8 heads N8192
// D128 / 112 161 -> 155, 16 heads N2048 D64 33 -> 31; before, the sums of all three filled the chip with whole groups, now
// those of two fill it with halves).
// The state slots of the group sums use the layout of the 16-bit kernels, so state_prefix_kernel serves both.
#pragma once
#include "cott_colscan.h"
#include "cott_terms.h"

namespace cott {

typedef ProblemT<float> ProblemF;
typedef ProblemSetT<float> ProblemSetF;

constexpr int kSplitChunk = 32;  // positions per chunk

template <int T>
struct SplitPairs;  // (a term, b term) of a product, smallest first; the last pair is hi hi
template <>
struct SplitPairs<2> {
    static constexpr int N = 3, A[3] = {1, 0, 0}, B[3] = {0, 1, 0};
};
template <>
struct SplitPairs<3> {
    static constexpr int N = 6, A[6] = {2, 0, 1, 1, 0, 0}, B[6] = {0, 2, 1, 0, 1, 0};
};

// One term of a [32][D] operand tile in LDS.
template <int D>
struct SplitTile {
    static constexpr int RS = D == 128 ? 128 : D + 16;
    static constexpr int SIZE = kSplitChunk * RS;
    __device__ static __forceinline__ int piece(int r, int c) {  // element offset of 16-byte piece c of row r
        return r * RS + 8 * (D == 128 ? wide_piece(r, c) : c);
    }
    // the same as an LDS address, from that of piece c < 4 to piece c + 4 ks (the turned pieces differ in two bits of the
    // address, tiles start at multiples of 256 bytes there: one instruction each time instead of a register for every ks)
    __device__ static __forceinline__ uint32_t step(uint32_t at, int ks) { return D == 128 ? at ^ (64u * ks) : at + 64u * ks; }
};

template <int DI, int DJ, int T, bool SUMS>
struct SplitTiling {
    static_assert(DI % 64 == 0 && DJ % 64 == 0, "four wavefronts of whole 16-column tiles");
    static constexpr int KS = DI / 32, NIT = DI / 16, NJT = DJ / 16, NJW = NJT / 4;
    static constexpr int AB = SplitTile<DI>::SIZE, C = SplitTile<DJ>::SIZE;
    static constexpr int SCORES = 2 * T * 2 * 64;  // u32x4: [2 buffers][T terms][2 position blocks][64]: keys of both key blocks
    static constexpr size_t LDS = ((SUMS ? 1 : 2) * AB + C) * 2 * T * sizeof(u16) + (SUMS ? 0 : SCORES * sizeof(u32x4));
    static constexpr int STATE_FLOATS = DI * DJ;
};

// LDS addresses in bytes.
typedef const __attribute__((address_space(3))) u16 *lds_ptr;
__device__ __forceinline__ uint32_t lds_address(const u16 *p) { return (uint32_t)(uintptr_t)(lds_ptr)p; }
__device__ __forceinline__ u32x4 lds_read16(uint32_t at) {
    return *reinterpret_cast<const __attribute__((address_space(3))) u32x4 *>((lds_ptr)(uintptr_t)at);
}
__device__ __forceinline__ u32x2 lds_read_tr16(uint32_t at) {
    s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)(uintptr_t)at);
    return bitcast<u32x2>(v);
}

// One operand of a problem: the rows of one head, fp32, or bf16 (an upstream gradient as the consumer of a bf16 output left
// it: exact as a hi part, so the tiles are those of the converted tensor; T = 2 only).
struct SplitRows {
    rsrc_t rs;
    uint32_t esz;  // bytes per element
    bool half;
};
__device__ __forceinline__ SplitRows split_rows(const float *base, size_t head, int half, int N, int ld, int d) {
    SplitRows s;
    s.half = half != 0;
    s.esz = s.half ? 2u : 4u;
    s.rs = make_rsrc_uniform(reinterpret_cast<const char *>(base) + head * s.esz, ((uint32_t)(N - 1) * ld + d) * s.esz);
    return s;
}

struct SplitRange {
    int N, nsteps, p0, p1, reversed;  // chunks of 32 positions p0 .. p1-1 in walking order
    __device__ __forceinline__ int first_row(int p) const { return (reversed ? nsteps - 1 - p : p) * kSplitChunk; }
};

typedef __attribute__((ext_vector_type(2))) unsigned short u16x2;
// How two fp32 numbers are split into T packed pairs of bf16 terms.  T = 2: rounded to nearest, 16 significant bits.  T = 3: the
// terms hold all 24 bits however they are chosen; what the six products leave out, mid lo + lo mid, is of either sign and
// below 2^-24 of a product of two rounded numbers, 1.5 2^-23 of a rounded and a cut one (two cut ones: 2^-21, always of the
// product's sign).  Every product has an operand from memory:
//   ROUNDED  operands from memory, each term the nearest bf16 number.
//   CUT      accumulators (state, scores), whose first term must not round up to infinity at the largest numbers.  (Rounding the
//            second one leaves the error as it is: 1.3e-7 at 1 x 4 x 2048 x 128.)
//   GUARDED  operand rows with a number whose nearest bf16 number is infinite: all terms cut, with the sign of the number.
//            `least` 0x0080, for rows with an infinite number: lower terms that are zero become the smallest normal number of that
//            sign, also those of the infinite number: an infinite factor then meets no exact zero among the other factor's lower
//            terms, and every partial product of inf * x is the infinity that inf * x is (and not a number, from the hi parts,
//            for x = 0).  To finite products that adds 2^-126 of a factor.
enum SplitMode { ROUNDED, CUT, GUARDED };
template <int T, SplitMode M>
__device__ __forceinline__ void split_pair(float a, float b, uint32_t *t, unsigned short least = 0) {
#pragma unroll
    for (int x = 0; x < T; ++x) {
        if ((T == 2 || M == ROUNDED) && x < 2)  // (the third is exact)
            t[x] = Bf16::pack2(a, b);
        else
            t[x] = __builtin_amdgcn_perm(bitcast<uint32_t>(b), bitcast<uint32_t>(a), 0x07060302u);
        if (x + 1 < T) {
            if constexpr (T == 2 || M == ROUNDED) {
                asm("" : "+v"(t[x]));  // (else the compiler rounds a once more by itself)
                a -= bitcast<float>(t[x] << 16);
                b -= bitcast<float>(t[x] & 0xffff0000u);
            } else {
                a -= bitcast<float>(bitcast<uint32_t>(a) & 0xffff0000u);
                b -= bitcast<float>(bitcast<uint32_t>(b) & 0xffff0000u);
                if (M == GUARDED && x == 0) {  // (inf - inf: the median of two non-numbers and zero is zero)
                    a = __builtin_amdgcn_fmed3f(a, a, 0.f);
                    b = __builtin_amdgcn_fmed3f(b, b, 0.f);
                }
            }
        }
        if constexpr (T == 3 && M == GUARDED) {
            if (x > 0) {
                const uint32_t some = bitcast<uint32_t>(__builtin_elementwise_max(bitcast<u16x2>(t[x]), u16x2{least, least}));
                t[x] = (some & 0x7fff7fffu) | (t[0] & 0x80008000u);
            }
        }
    }
}
// four accumulator values -> T pairs of dwords
template <int T>
__device__ __forceinline__ void split_acc(f32x4 v, u32x2 *t) {
    uint32_t a[T], b[T];
    split_pair<T, CUT>(v[0], v[1], a);
    split_pair<T, CUT>(v[2], v[3], b);
#pragma unroll
    for (int x = 0; x < T; ++x) t[x] = u32x2{a[x], b[x]};
}

// Loader role: 256 threads move the tiles two chunks ahead and form the scores of the chunk the compute wavefronts are at.
template <int DI, int DJ, int T, bool SUMS>
__device__ __forceinline__ void split_loader_role(const SplitRows &rA, const SplitRows &rB, const SplitRows &rC, int di, int dj,
                                                 int lda, int ldb, int ldc, const SplitRange &r, int tid, u16 *sA, u16 *sB, u16 *sC,
                                                 u32x2 *sP) {
    using TL = SplitTiling<DI, DJ, T, SUMS>;
    constexpr int PF = 2, PI = kSplitChunk * DI / 8 / 256, PJ = kSplitChunk * DJ / 8 / 256;
    static_assert(PI >= 1 && PJ >= 1, "a piece per loader thread at least");
    const int l = tid & 63, g = l >> 4, m = l & 15;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    u32x4 ra[PF][SUMS ? 1 : PI][2], rb[PF][PI][2], rc[PF][PJ][2];
    // Piece u of this thread in a tile of D columns: wavefront w holds rows 8w .. 8w+7 of every operand.
    auto piece_row = [&](int u, int D) __attribute__((always_inline)) { return 8 * w + (64 * u + l) / (D / 8); };
    auto piece_col = [&](int D) __attribute__((always_inline)) { return l % (D / 8); };
    // Byte offsets of the pieces within their chunk; out of range, so that they load zeros, for columns past the runtime width.
    uint32_t offA[PI], offB[PI], offC[PJ];
#pragma unroll
    for (int u = 0; u < PI; ++u) {
        const int row = piece_row(u, DI), col = 8 * piece_col(DI);
        offA[u] = col < di ? (uint32_t)(row * lda + col) * rA.esz : kOobOffset;
        offB[u] = col < di ? (uint32_t)(row * ldb + col) * rB.esz : kOobOffset;
    }
#pragma unroll
    for (int u = 0; u < PJ; ++u) {
        const int row = piece_row(u, DJ), col = 8 * piece_col(DJ);
        offC[u] = col < dj ? (uint32_t)(row * ldc + col) * rC.esz : kOobOffset;
    }
    auto load_piece = [&](u32x4 *x, const SplitRows &src, uint32_t off) __attribute__((always_inline)) {
        x[0] = buf_load16(src.rs, off);
        x[1] = buf_load16(src.rs, T == 2 && src.half ? kOobOffset : off + 16u);  // (bf16 rows: as many loads in flight)
    };
    auto load_chunk = [&](int s, int p) __attribute__((always_inline)) {
        const uint32_t row0 = (uint32_t)r.first_row(min(p, r.p1 - 1));
        const uint32_t a0 = row0 * lda * rA.esz, b0 = row0 * ldb * rB.esz, c0 = row0 * ldc * rC.esz;
#pragma unroll
        for (int u = 0; u < PI; ++u) {
            if constexpr (!SUMS) load_piece(ra[s][u], rA, offA[u] + a0);
            load_piece(rb[s][u], rB, offB[u] + b0);
        }
#pragma unroll
        for (int u = 0; u < PJ; ++u) load_piece(rc[s][u], rC, offC[u] + c0);
    };
    // one piece -> its T tiles; largest: the largest magnitude seen so far
    auto stage_piece = [&](u16 *tile, int term_stride, const u32x4 *x, const SplitRows &src, int at, auto mode, unsigned short least,
                           float &largest) __attribute__((always_inline)) {
        constexpr SplitMode M = decltype(mode)::value;
        u32x4 t[T];
        if (T == 2 && src.half) {
            t[0] = x[0];
            t[1] = u32x4{0u, 0u, 0u, 0u};
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                uint32_t q[T];
                const float a = bitcast<float>(x[e >> 1][2 * (e & 1)]), b = bitcast<float>(x[e >> 1][2 * (e & 1) + 1]);
                split_pair<T, M>(a, b, q, least);
#pragma unroll
                for (int y = 0; y < T; ++y) t[y][e] = q[y];
                if constexpr (T == 3 && M == ROUNDED)
                    largest = __builtin_fmaxf(__builtin_fmaxf(largest, __builtin_fabsf(a)), __builtin_fabsf(b));
            }
        }
#pragma unroll
        for (int e = 0; e < T; ++e) *reinterpret_cast<u32x4 *>(tile + e * term_stride + at) = t[e];
    };
    auto stage_a = [&](int s, int buf, auto mode, float &largest) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < PI; ++u)
            stage_piece(sA + buf * TL::AB, 2 * TL::AB, ra[s][u], rA, SplitTile<DI>::piece(piece_row(u, DI), piece_col(DI)), mode, 0, largest);
    };
    auto stage_bc = [&](int s, int buf, auto mode, unsigned short least, float &largest) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < PI; ++u)
            stage_piece(sB + buf * TL::AB, 2 * TL::AB, rb[s][u], rB, SplitTile<DI>::piece(piece_row(u, DI), piece_col(DI)), mode, least, largest);
#pragma unroll
        for (int u = 0; u < PJ; ++u)
            stage_piece(sC + buf * TL::C, 2 * TL::C, rc[s][u], rC, SplitTile<DJ>::piece(piece_row(u, DJ), piece_col(DJ)), mode, least, largest);
    };
    auto stage = [&](int s, int buf) __attribute__((always_inline)) {
        constexpr std::integral_constant<SplitMode, ROUNDED> rounded{};
        constexpr std::integral_constant<SplitMode, GUARDED> guarded{};
        float largest = 0.f;
        if constexpr (!SUMS) stage_a(s, buf, rounded, largest);
        stage_bc(s, buf, rounded, 0, largest);
        if constexpr (T == 3) {
            // a number that the nearest bf16 one to is infinite (this wavefront holds the same rows of all operands): once more
            if (__any(largest >= bitcast<float>(0x7f7f8000u))) {
                if constexpr (!SUMS) stage_a(s, buf, guarded, largest);
                // (infinite entries of A need nothing else: they enter outputs only, see add_rest)
                bool inf = false;
                auto look = [&](const u32x4 *x) __attribute__((always_inline)) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) inf |= (x[e >> 2][e & 3] & 0x7fffffffu) == 0x7f800000u;
                };
#pragma unroll
                for (int u = 0; u < PI; ++u) look(rb[s][u]);
#pragma unroll
                for (int u = 0; u < PJ; ++u) look(rc[s][u]);
                stage_bc(s, buf, guarded, __any(inf) ? 0x0080 : 0, largest);
            }
        }
    };
    // Score tile of this wavefront (0..2): key block kt against position block pb, transposed (a lane holds four
    // consecutive keys of one position).  Sum over the past: (0,0) (1,0) (1,1); over the future: (0,0) (0,1) (1,1).
    const int pb = r.reversed ? (w == 2) : (w >= 1), kt = r.reversed ? (w >= 1) : (w == 2);
    const int dir = pb != kt ? 0 : (r.reversed ? 1 : -1), side = dir * (4 * g - m);
    auto scores = [&](int buf) __attribute__((always_inline)) {
        if (w >= 3) return;
        // T = 3: two accumulators for the leading products, half the chain of sums that are cut to fp32.  (From the last columns to
        // the first: the order is free and decides how nearly cancelling scores round; with this one those that the tests look
        // at by themselves keep to 8e-7.)
        constexpr int CH = T == 3 ? 2 : 1;
        const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
        f32x4 hi[CH], rest[2] = {zero, zero};
#pragma unroll
        for (int c = 0; c < CH; ++c) hi[c] = zero;
#pragma unroll
        for (int step = 0; step < TL::KS; ++step) {
            const int ks = T == 3 ? TL::KS - 1 - step : step;
            u32x4 a[T], b[T];
#pragma unroll
            for (int x = 0; x < T; ++x) {
                a[x] = ld128(sB + (2 * x + buf) * TL::AB + 16 * kt * SplitTile<DI>::RS + SplitTile<DI>::piece(m, 4 * ks + g));
                b[x] = ld128(sA + (2 * x + buf) * TL::AB + 16 * pb * SplitTile<DI>::RS + SplitTile<DI>::piece(m, 4 * ks + g));
            }
#pragma unroll
            for (int e = 0; e + 1 < SplitPairs<T>::N; ++e)
                rest[e & 1] = Bf16::mfma(a[SplitPairs<T>::A[e]], b[SplitPairs<T>::B[e]], rest[e & 1]);
            hi[ks % CH] = Bf16::mfma(a[0], b[0], hi[ks % CH]);
        }
        f32x4 main = hi[0];
        if constexpr (CH == 2) main += hi[1];
        f32x4 acc = main + (rest[0] + rest[1]);
        if (T == 3 && __any(any_nan(acc))) acc = number_or(acc, main);
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[q] = side + dir * q >= 0 ? acc[q] : 0.f;
        u32x2 t[T];
        split_acc<T>(acc, t);
#pragma unroll
        for (int x = 0; x < T; ++x) sP[((buf * T + x) * 2 + pb) * 128 + 2 * l + kt] = t[x];
    };
#pragma unroll
    for (int s = 0; s < PF; ++s) load_chunk(s, r.p0 + s);
    stage(0, 0);
    load_chunk(0, r.p0 + PF);
    __syncthreads();
    run_rounds<PF>(r.p0, r.p1, [&](int s, int p) __attribute__((always_inline)) {
        const int s1 = (s + 1) % PF, buf = s;  // (PF = 2: the LDS buffer is the register stage)
        if constexpr (!SUMS) scores(buf);
        stage(s1, buf ^ 1);
        load_chunk(s1, p + 1 + PF);
        chunk_barrier();
    });
}

// the bf16 matrix instruction over 16 instead of 32 contraction steps, four of them per lane
__device__ __forceinline__ f32x4 mfma_half(u32x2 a, u32x2 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(bitcast<s16x4>(a), bitcast<s16x4>(b), c, 0, 0, 0);
}

// Compute role: wavefront w of 4 owns column tiles NJW * w .. of the state (all rows, interleaved as in colscan_kernel) and
// of the output.
template <int DI, int DJ, int T, bool SUMS, bool FUT>
__device__ __forceinline__ void split_compute_role(const ColStateIO &io, float *O_head, int ldo, int di, int dj, const SplitRange &r,
                                                  int w, int l, const u16 *sA, const u16 *sB, const u16 *sC, const u32x4 *sP) {
    using TL = SplitTiling<DI, DJ, T, SUMS>;
    using TP = SplitPairs<T>;
    constexpr int KS = TL::KS, NIT = TL::NIT, NJW = TL::NJW;
    const int g = l >> 4, m = l & 15;
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    const rsrc_t rO = make_rsrc_uniform(O_head, SUMS ? 0u : ((uint32_t)(r.N - 1) * ldo + dj) * 4u);
    f32x4 S[NIT][NJW];
#pragma unroll
    for (int it = 0; it < NIT; ++it)
#pragma unroll
        for (int jw = 0; jw < NJW; ++jw) S[it][jw] = zero;
    // slot of the standard tile layout that holds this lane's four rows of S[it][jw]
    auto slot_at = [&](int it, int jw) __attribute__((always_inline)) {
        return (size_t)((2 * (it >> 1) + (g >> 1)) * TL::NJT + NJW * w + jw) * 64 + 16 * (2 * (g & 1) + (it & 1)) + m;
    };
    if (!SUMS && io.seed != nullptr) {
        const f32x4 *gs = reinterpret_cast<const f32x4 *>(io.seed);
#pragma unroll
        for (int it = 0; it < NIT; ++it)
#pragma unroll
            for (int jw = 0; jw < NJW; ++jw) S[it][jw] = gs[slot_at(it, jw)];
    }
    if (!SUMS && DI == DJ && io.seed_t != nullptr) {  // the twin's slot, transposed: this lane's four rows are four of its columns
#pragma unroll
        for (int it = 0; it < NIT; ++it)
#pragma unroll
            for (int jw = 0; jw < NJW; ++jw)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    S[it][jw][q] = io.seed_t[(((NJW * w + jw) * TL::NJT + 2 * (it >> 1) + (g >> 1)) * 64 + 16 * (m >> 2) +
                                              8 * (g & 1) + 4 * (it & 1) + q) * 4 + (m & 3)];
    }
    if (!SUMS && io.sin != nullptr) {
#pragma unroll
        for (int it = 0; it < NIT; ++it)
#pragma unroll
            for (int jw = 0; jw < NJW; ++jw)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int i = 32 * (it >> 1) + 8 * g + 4 * (it & 1) + q, j = 16 * (NJW * w + jw) + m;
                    if (i < di && j < dj) S[it][jw][q] += io.sin[(size_t)i * io.lds + j];
                }
    }
    // C fragments of the chunk: keys 4g .. 4g+3 and 16+4g .. of column 16 (NJW w + jw) + m, the order of the score operands;
    // the state update contracts in the same order.
    u32x4 cf[NJW][T];
    f32x4 o[2][NJW];
    uint32_t a_at = lds_address(sA + SplitTile<DI>::piece(m, g)), b_at[2], c_at[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int row = 16 * h + 4 * g + (m >> 2);
        b_at[h] = lds_address(sB + SplitTile<DI>::piece(row, m & 3));
        c_at[h] = lds_address(sC + SplitTile<DJ>::piece(row, 2 * NJW * w + ((m >> 1) & 1)) + 4 * (m & 1));
    }
    // C tiles: column tile jw, two pieces on, of this wavefront (with one tile there is none)
    auto c_step = [&](uint32_t at, int jw) __attribute__((always_inline)) { return DJ == 128 ? at ^ (32u * jw) : at; };
    // this lane's four output columns of the first column tile in the first row of a chunk; dj is a multiple of 16, so that a
    // column tile lies inside the width or outside as a whole
    const uint32_t o_at = (uint32_t)(m * ldo + 16 * NJW * w + 4 * g) * 4u;
    // v = hi + rest; T = 3: where that is no number, hi, which has the value of the single-number arithmetic (a rest of inf -
    // inf or inf * 0).  The empty asm keeps the repair behind its branch: as selects it would take 40 instructions a chunk.
    auto add_rest = [&](f32x4 (&v)[2][NJW], const f32x4 (&hi)[2][NJW], const f32x4 (&rest)[2][NJW]) __attribute__((always_inline)) {
        f32x4 sum = zero;
#pragma unroll
        for (int pb = 0; pb < 2; ++pb)
#pragma unroll
            for (int jw = 0; jw < NJW; ++jw) {
                v[pb][jw] = hi[pb][jw] + rest[pb][jw];
                if constexpr (T == 3) sum += v[pb][jw];
            }
        if constexpr (T == 3) {
            if (__any(any_nan(sum))) {
                asm volatile("" ::: "memory");
#pragma unroll
                for (int pb = 0; pb < 2; ++pb)
#pragma unroll
                    for (int jw = 0; jw < NJW; ++jw) v[pb][jw] = number_or(v[pb][jw], hi[pb][jw]);
            }
        }
    };
    auto finish = [&](int buf, int p) __attribute__((always_inline)) {
        const int row0 = r.first_row(p);
        u32x4 pf[2][T];
#pragma unroll
        for (int x = 0; x < T; ++x)
#pragma unroll
            for (int pb = 0; pb < 2; ++pb) pf[pb][x] = sP[((buf * T + x) * 2 + pb) * 64 + l];
        f32x4 rest[2][NJW];
#pragma unroll
        for (int pb = 0; pb < 2; ++pb)
#pragma unroll
            for (int jw = 0; jw < NJW; ++jw) rest[pb][jw] = zero;
#pragma unroll
        for (int e = 0; e < TP::N; ++e)
#pragma unroll
            for (int pb = 0; pb < 2; ++pb)
#pragma unroll
                for (int jw = 0; jw < NJW; ++jw) {
                    f32x4 &acc = e + 1 < TP::N ? rest[pb][jw] : o[pb][jw];
                    const u32x4 c = cf[jw][TP::A[e]], q = pf[pb][TP::B[e]];
                    // one position block has a single live key block: the other's keys stay out (a masked zero times an
                    // infinite entry of C would be no number)
                    if (pb == (FUT ? 1 : 0))
                        acc = mfma_half(FUT ? u32x2{c[2], c[3]} : u32x2{c[0], c[1]}, FUT ? u32x2{q[2], q[3]} : u32x2{q[0], q[1]}, acc);
                    else
                        acc = Bf16::mfma(c, q, acc);
                }
        f32x4 v[2][NJW];
        add_rest(v, o, rest);
#pragma unroll
        for (int pb = 0; pb < 2; ++pb)
#pragma unroll
            for (int jw = 0; jw < NJW; ++jw)
            {
                const uint32_t tile = 16 * (NJW * w + jw) < dj ? (uint32_t)(row0 + 16 * pb) * ldo * 4u + 64u * jw : kOobOffset;
                __builtin_amdgcn_raw_buffer_store_b128(bitcast<u32x4>(v[pb][jw]), rO, (int)(o_at + tile), 0, 0);
            }
    };
    u32x4 s[NJW][T];  // terms of the state rows of the next contraction step
    auto pack_state = [&](int ks, int jw) __attribute__((always_inline)) {
        u32x2 lo[T], hi[T];
        split_acc<T>(S[2 * ks][jw], lo);
        split_acc<T>(S[2 * ks + 1][jw], hi);
#pragma unroll
        for (int x = 0; x < T; ++x) s[jw][x] = cat(lo[x], hi[x]);
    };
    // keeps the terms of the next chunk's first rows where they are formed, under this chunk's last products
    auto pin_state = [&](int jw) __attribute__((always_inline)) {
#pragma unroll
        for (int x = 0; x < T; ++x) asm volatile("" : "+v"(s[jw][x]));
    };
    auto chunk = [&](int buf) __attribute__((always_inline)) {
        f32x4 ah[2][NJW], ar[2][NJW];
#pragma unroll
        for (int pb = 0; pb < 2; ++pb)
#pragma unroll
            for (int jw = 0; jw < NJW; ++jw) ah[pb][jw] = ar[pb][jw] = zero;
        u32x4 a[2][T], b[2][T];
        // (else the addresses of all steps would be kept in registers)
        asm volatile("" : "+v"(a_at), "+v"(b_at[0]), "+v"(b_at[1]), "+v"(c_at[0]), "+v"(c_at[1]));
        auto read_a = [&](int ks) __attribute__((always_inline)) {
#pragma unroll
            for (int pb = 0; pb < 2; ++pb)
#pragma unroll
                for (int x = 0; x < T; ++x) a[pb][x] = lds_read16(SplitTile<DI>::step(a_at, ks) + 2 * ((2 * x + buf) * TL::AB + 16 * pb * SplitTile<DI>::RS));
        };
        auto read_b = [&](int ks) __attribute__((always_inline)) {
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int x = 0; x < T; ++x)
                    b[t][x] = cat(lds_read_tr16(SplitTile<DI>::step(b_at[0], ks) + 2 * ((2 * x + buf) * TL::AB + 4 * t)),
                                  lds_read_tr16(SplitTile<DI>::step(b_at[1], ks) + 2 * ((2 * x + buf) * TL::AB + 4 * t)));
        };
        auto state_product = [&](int jw) __attribute__((always_inline)) {
#pragma unroll
            for (int e = 0; e < TP::N; ++e)
#pragma unroll
                for (int pb = 0; pb < 2; ++pb) {
                    if (e + 1 < TP::N)
                        ar[pb][jw] = Bf16::mfma(s[jw][TP::A[e]], a[pb][TP::B[e]], ar[pb][jw]);
                    else
                        ah[pb][jw] = Bf16::mfma(s[jw][0], a[pb][0], ah[pb][jw]);
                }
        };
        // S += B^T C of one contraction step.  T = 3: the product of the chunk by itself first, one addition (rounded to
        // nearest) to the state then; accumulating the six partial products on the state itself loses a bit over long sums.
        auto update = [&](int ks, int t) __attribute__((always_inline)) {
            {
                f32x4 d[NJW];
#pragma unroll
                for (int e = 0; e < TP::N; ++e)
#pragma unroll
                    for (int jw = 0; jw < NJW; ++jw)
                        d[jw] = Bf16::mfma(b[t][TP::A[e]], cf[jw][TP::B[e]], e > 0 ? d[jw] : (T == 3 ? zero : S[2 * ks + t][jw]));
#pragma unroll
                for (int jw = 0; jw < NJW; ++jw) S[2 * ks + t][jw] = T == 3 ? S[2 * ks + t][jw] + d[jw] : d[jw];
            }
        };
        // Under the products of one kind the operands of the other are read and split.
        if constexpr (!SUMS) {
            read_a(0);
        } else {
            read_b(0);
        }
#pragma unroll
        for (int jw = 0; jw < NJW; ++jw)
#pragma unroll
            for (int x = 0; x < T; ++x)
                cf[jw][x] = cat(lds_read_tr16(c_step(c_at[0], jw) + 2 * (2 * x + buf) * TL::C), lds_read_tr16(c_step(c_at[1], jw) + 2 * (2 * x + buf) * TL::C));
        sched_fence();
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            if constexpr (!SUMS) {
                // a matrix instruction, and under it vector ones and a read of LDS
                auto interleave = [&](auto n, auto vector) __attribute__((always_inline)) {
#pragma unroll
                    for (int e = 0; e < decltype(n)::value; ++e) {
                        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(0x2, decltype(vector)::value, 0);
                        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                    }
                };
                read_b(ks);
                state_product(0);
                sched_fence();
                constexpr std::integral_constant<int, NJW * TP::N> half{};
                if constexpr (NJW == 2) {
                    pack_state((ks + 1) % KS, 0);  // (the first step's rows are final after its own update)
                    if (ks + 1 == KS) pin_state(0);
                    state_product(1);
                    interleave(half, std::integral_constant<int, 4>{});
                    sched_fence();
                }
                pack_state((ks + 1) % KS, NJW - 1);
                if (ks + 1 == KS) pin_state(NJW - 1);
                update(ks, 0);
                interleave(half, std::integral_constant<int, 4>{});
                sched_fence();
                if (ks + 1 < KS) read_a(ks + 1);
                update(ks, 1);
                interleave(half, std::integral_constant<int, 2>{});
                sched_fence();
            } else {
                update(ks, 0);
                update(ks, 1);
                if (ks + 1 < KS) read_b(ks + 1);
            }
        }
        if constexpr (!SUMS) {
            add_rest(o, ah, ar);
        }
    };
    if constexpr (!SUMS) {
#pragma unroll
        for (int jw = 0; jw < NJW; ++jw) pack_state(0, jw);
    }
    __syncthreads();
    run_rounds<2>(r.p0, r.p1, [&](int buf, int p) __attribute__((always_inline)) {
        if constexpr (!SUMS) {
            if (p > r.p0) finish(buf ^ 1, p - 1);
        }
        chunk(buf);
        chunk_barrier();
    });
    if constexpr (SUMS) {
        f32x4 *slot = reinterpret_cast<f32x4 *>(io.sums);
#pragma unroll
        for (int it = 0; it < NIT; ++it)
#pragma unroll
            for (int jw = 0; jw < NJW; ++jw) slot[slot_at(it, jw)] = S[it][jw];
        return;
    }
    if (r.p1 > r.p0) finish((r.p1 - 1 - r.p0) & 1, r.p1 - 1);
    if (io.sout != nullptr) {
#pragma unroll
        for (int it = 0; it < NIT; ++it)
#pragma unroll
            for (int jw = 0; jw < NJW; ++jw)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int i = 32 * (it >> 1) + 8 * g + 4 * (it & 1) + q, j = 16 * (NJW * w + jw) + m;
                    if (i < di && j < dj) io.sout[(size_t)i * io.lds + j] = S[it][jw][q];
                }
    }
}

// 512 threads: wavefronts 0..3 compute, 4..7 load.  Grid: grid_for(BH, count, G) for the scan, grid_for(BH, nact * sub,
// G - 1) for the sums of the groups.  spg: chunks of 32 positions per group.
template <int DI, int DJ, int T, bool SUMS>
__global__ __launch_bounds__(512, T == 2 ? 4 : 2) void split_scan_kernel(ProblemSetF set, int BH, int N, int nsteps, int spg, int G) {
    using TL = SplitTiling<DI, DJ, T, SUMS>;
    __shared__ __attribute__((aligned(256))) unsigned char smem[TL::LDS];  // (see SplitTile::step)
    u16 *sB = reinterpret_cast<u16 *>(smem), *sC = sB + 2 * T * TL::AB, *sA = sC + 2 * T * TL::C;
    u32x4 *sP = reinterpret_cast<u32x4 *>(sA + (SUMS ? 0 : 2 * T * TL::AB));
    const int l = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int sub = set.sub;
    const WorkItem wi = decode_workgroup(SUMS ? set.nact * sub : set.count, BH, set.xcds);
    if (wi.grp >= (SUMS ? G - 1 : G)) return;
    const ProblemF &pr = set.p[SUMS ? set.act[wi.prob / sub] : wi.prob];
    const int di = pr.di, dj = pr.dj;
    SplitRange r;
    r.N = N;
    r.nsteps = nsteps;
    r.p0 = wi.grp * spg;
    r.p1 = min(r.p0 + spg, nsteps);
    r.reversed = pr.reversed;
    ColStateIO io;
    if constexpr (SUMS) {  // a piece of the group; one past its end leaves a zero slot
        const int piece = wi.prob % sub, per = (spg + sub - 1) / sub;
        r.p0 += piece * per;
        r.p1 = min(r.p0 + per, r.p1);
        io.sums = pr.gstate + (((size_t)wi.bh * G + wi.grp) * sub + piece) * TL::STATE_FLOATS;
        if (r.p1 <= r.p0) {
            for (int e = threadIdx.x; e < TL::STATE_FLOATS / 4; e += 512) reinterpret_cast<f32x4 *>(io.sums)[e] = f32x4{0.f, 0.f, 0.f, 0.f};
            return;
        }
    } else {
        const size_t slot = ((size_t)wi.bh * G + wi.grp) * sub * TL::STATE_FLOATS;
        if (pr.seed_from >= 0) {
            if (set.p[pr.seed_from].gstate != nullptr) io.seed_t = set.p[pr.seed_from].gstate + slot;
        } else if (pr.gstate != nullptr) {
            io.seed = pr.gstate + slot;
        }
        if (pr.sin != nullptr) io.sin = pr.sin + (size_t)wi.bh * di * pr.lds;
        if (pr.sout != nullptr && wi.grp == G - 1) io.sout = pr.sout + (size_t)wi.bh * di * pr.lds;
        io.lds = pr.lds;
    }
    if (wv >= 4) {
        const SplitRows rA = split_rows(pr.A, head_base(pr.bsA, pr.hsA, pr.H, wi.bh), pr.bf16_operands & 1, N, pr.lda, di);
        const SplitRows rB = split_rows(pr.B, head_base(pr.bsB, pr.hsB, pr.H, wi.bh), pr.bf16_operands & 2, N, pr.ldb, di);
        const SplitRows rC = split_rows(pr.C, head_base(pr.bsC, pr.hsC, pr.H, wi.bh), pr.bf16_operands & 4, N, pr.ldc, dj);
        split_loader_role<DI, DJ, T, SUMS>(rA, rB, rC, di, dj, pr.lda, pr.ldb, pr.ldc, r, (int)threadIdx.x - 256, sA, sB, sC,
                                          reinterpret_cast<u32x2 *>(sP));
    } else {
        float *O_head = SUMS ? nullptr : pr.O + head_base(pr.bsO, pr.hsO, pr.H, wi.bh);
        if (!SUMS && pr.reversed)
            split_compute_role<DI, DJ, T, SUMS, true>(io, O_head, pr.ldo, di, dj, r, wv, l, sA, sB, sC, sP);
        else
            split_compute_role<DI, DJ, T, SUMS, false>(io, O_head, pr.ldo, di, dj, r, wv, l, sA, sB, sC, sP);
    }
}

}  // namespace cott
