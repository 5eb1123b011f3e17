// Chunked causal scan for 16-bit tensors whose head dims lie outside the kernels of cott_mfma.h (wider than 128
// columns, up to 256 contracted ones; value widths are cut into slices, so any multiple of 16).
//
//     out_c = ((A_c B_c^T) o mask) C_c + A_c S_c ;   S_{c+1} = S_c + B_c^T C_c          (chunks of 32 positions)
//
// One workgroup walks the sequence of one head for one 64-column slice of C and of the output.
//   * Eight compute wavefronts each own 16 columns and half of the DI rows of the state in fp32 accumulators (32
//     registers at DI = 256).  The two halves of a column exchange partial outputs through LDS: each finishes one of
//     the chunk's two blocks of 16 positions.  The rows of neighbouring 16 x 16 tiles are interleaved as in colscan_kernel (tile 2ks+t, row 4g+q
//     holds state row 32ks+8g+4t+q), which makes a lane's accumulators eight consecutive contraction steps: they are
//     the operand of A_c S_c as they lie and the state never passes through LDS.
//   * Four loader wavefronts move the tiles global -> registers -> LDS two chunks ahead, form the three live 16 x 16
//     score tiles of the chunk (once per workgroup, handed to the compute wavefronts through LDS) and write the
//     finished output tile to memory as 16-byte pieces of whole 128-byte row segments.
//   * One barrier per chunk: the product of the scores with C_c is finished at the start of the next chunk.
// Precision: the plain-FMA kernel that served these widths keeps state and scores in fp32, with 24 significant bits.
// Here both enter the matrix instructions as the sum of three 16-bit numbers that holds all of them (split3), so that
// every product is that of the fp32 number and what is left is the order of the fp32 sums.  fp16: the state is scaled by
// a power of two per column first, so that neither its largest nor its small entries leave the range, and the scores and
// C take part as bf16 triples and pairs (C exactly).
// What bounds it: the chain of chunks, 1.4 us each at DI = 256, and in it the vector instructions of the splits (with two
// terms, 16 significant bits, it took 1.27 us).  Each contraction step's LDS reads and splits are issued between the matrix
// instructions of the step before: left to itself the compiler put a step's reads, its splits and its products one after
// the other (bf16, same results: 16 heads N1024 D256 forward 31.0 -> 30.3 us, gradients 61.5 -> 60.0; 2 heads N4096 38.4 ->
// 37.2 and 50.5 -> 48.6; 16 heads N1000 D224 29.8 -> 28.6 and 57.5 -> 55.2; fp16 1 %).  64-column slices rather than 128:
// twice as many workgroups share the chip, and with few heads workgroups are what is short; the rest of the chip is filled
// by sequence groups (wide_groups).  B1 H16 N1024 D256: forward 30 us, gradients (192 workgroups, whole sequences) 60 us
// with their passes, where the plain-FMA kernel took 18.0 ms for both.  Share of the outputs that are not the 16-bit number
// nearest to the exact result, same shape: 1.5e-4 (bf16) and 1.2e-3 (fp16), plain-FMA kernel 2.9e-4 and 3.2e-3, two terms
// 2.4e-3 and 5.5e-3.
#pragma once
#include "cott_mfma.h"
#include "cott_terms.h"

namespace cott {

constexpr int kWideChunk = 32;  // positions per chunk: with 64 the double-buffered 256-wide tiles do not fit LDS
constexpr int kWideSlice = 64;  // output columns per workgroup
constexpr int kWideCompute = 8, kWideLoad = 4;  // wavefronts of either role

struct WideOp {
    const u16 *A, *B, *C;  // (BH,N,di), (BH,N,di), (BH,N,dj)
    u16 *O;                // (BH,N,dj)
    const float *sin;      // (BH,di,dj) fp32 state to start from, or null
    float *sout;           // receives the state after the last position, or null
    int di, dj, reversed, slices;
};
struct WideSet {
    WideOp op[3];
    int count, items;  // ops; workgroups per head and group = all slices of all ops
    int xcds;
    // Few heads: the sequence is cut into G groups of cpg chunks (in walking order).  wide_scan_kernel<..., SUMS> leaves the
    // sum of B^T C over each group but the last in slots [head][item][1 + group] of wide_slot_vectors() float4 and, where
    // there is one, the start state in slot 0 (its workgroups `G - 1`; first_slot = 0, else 1); a group of the scan starts
    // from the sum of the slots up to its own number.  The scan itself then reads no sin: sout may be the same memory, and
    // the last group may write it before another one starts.
    int G, cpg, first_slot;
    f32x4 *slots;
};
// One slice's state in the order of its owners: [wavefront][tile][lane].
__host__ __device__ constexpr int wide_slot_vectors(int DI) { return DI * kWideSlice / 4; }
struct WideRange {
    int N, nchunks, p0, p1;  // chunks p0 .. p1-1 in walking order
};

template <int DI>
struct WideTiling {
    static_assert(DI % 64 == 0, "contracted dim padded to a multiple of 64");
    // LDS row stride (elements) of the A and B tiles: whole 256-byte spans, in which the 16-byte pieces of a row are
    // permuted (wide_piece)
    static constexpr int RS = (DI + 127) / 128 * 128;
    static constexpr int CS = kWideSlice + 16;
    static constexpr int OS = kWideSlice + 8;
    static constexpr int KS = DI / 32;
    static constexpr int TILE = kWideChunk * RS, CTILE = kWideChunk * CS, OTILE = kWideChunk * OS;
    static constexpr int PIECES = kWideChunk * DI / 8 / 256;  // 16-byte pieces of an A or B tile per loader thread
    // A and B tiles, C tiles, output tiles (two buffers each), then the score operands [2 buffers][hi, mid, lo][2 blocks]
    // [64] and the partial outputs [2 buffers][8 wavefronts][64]
    static constexpr int SCORES = 2 * 3 * 2 * 64;
    static constexpr size_t LDS = (4 * TILE + 2 * CTILE + 2 * OTILE) * sizeof(u16) +
                                  (SCORES + 2 * kWideCompute * 64) * sizeof(u32x4);
};

// eight fp16 numbers -> the same eight as bf16 hi + lo (exact: 8 + 8 significant bits hold the 11)
__device__ __forceinline__ void fp16_as_bf16_pair(u32x4 v, u32x4 &hi, u32x4 &lo) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float a = Fp16::to_float((u16)(v[e] & 0xffffu)), b = Fp16::to_float((u16)(v[e] >> 16));
        hi[e] = cut2<Bf16>(a, b);
        lo[e] = cut2<Bf16>(a - Bf16::to_float((u16)(hi[e] & 0xffffu)), b - Bf16::to_float((u16)(hi[e] >> 16)));
    }
}

template <class TR, int DI, bool SUMS>
__device__ __forceinline__ void wide_loader_role(const WideOp &op, int bh, int c0, const WideRange &rg, int tid, u16 *sA,
                                                 u16 *sB, u16 *sC, const u16 *sO, u32x2 *sP) {
    using T = WideTiling<DI>;
    constexpr int PF = 2, PIECES = T::PIECES;
    const int l = tid & 63, g = l >> 4, m = l & 15;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int di = op.di, dj = op.dj, reversed = op.reversed;
    const int N = rg.N, p0 = rg.p0, p1 = rg.p1;
    const uint32_t rows = (uint32_t)(N - 1);
    const rsrc_t rA = make_rsrc_uniform(op.A + (size_t)bh * N * di, (rows * di + di) * 2u);
    const rsrc_t rB = make_rsrc_uniform(op.B + (size_t)bh * N * di, (rows * di + di) * 2u);
    const rsrc_t rC = make_rsrc_uniform(op.C + (size_t)bh * N * dj + c0, (rows * dj + (dj - c0)) * 2u);
    const rsrc_t rO = make_rsrc_uniform(op.O + (size_t)bh * N * dj + c0, (rows * dj + (dj - c0)) * 2u);
    u32x4 ra[PF][PIECES], rb[PF][PIECES], rc[PF];
    const int ccol = (tid % (kWideSlice / 8)) * 8, crow = tid / (kWideSlice / 8);
    auto first_row = [&](int p) __attribute__((always_inline)) { return (reversed ? rg.nchunks - 1 - p : p) * kWideChunk; };
    auto load_chunk = [&](int s, int p) __attribute__((always_inline)) {
        const int row0 = first_row(min(p, p1 - 1));
#pragma unroll
        for (int u = 0; u < PIECES; ++u) {
            const int v = tid + 256 * u;
            const uint32_t off = (uint32_t)((row0 + v / (DI / 8)) * di + (v % (DI / 8)) * 8) * 2u;
            if constexpr (!SUMS) ra[s][u] = buf_load16(rA, off);
            rb[s][u] = buf_load16(rB, off);
        }
        rc[s] = buf_load16(rC, (uint32_t)((row0 + crow) * dj + ccol) * 2u);
    };
    auto stage = [&](int s, int buf) __attribute__((always_inline)) {
        const u32x4 z = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int u = 0; u < PIECES; ++u) {
            const int v = tid + 256 * u, col = (v % (DI / 8)) * 8, row = v / (DI / 8);
            const int at = row * T::RS + 8 * wide_piece(row, col / 8);
            if constexpr (!SUMS) *reinterpret_cast<u32x4 *>(sA + buf * T::TILE + at) = col < di ? ra[s][u] : z;
            *reinterpret_cast<u32x4 *>(sB + buf * T::TILE + at) = col < di ? rb[s][u] : z;
        }
        *reinterpret_cast<u32x4 *>(sC + buf * T::CTILE + crow * T::CS + ccol) = c0 + ccol < dj ? rc[s] : z;
    };
    // Score tile of this wavefront: key block kt against position block pb, transposed (a lane holds four consecutive
    // keys of one position).  Sum over the past: (0,0) (1,0) (1,1); over the future: (0,0) (0,1) (1,1).
    const int pb = reversed ? (w == 2) : (w >= 1), kt = reversed ? (w >= 1) : (w == 2);
    // key 4g+q of the tile counts for position m where side + dir q >= 0: on the diagonal the keys of its side, else all
    const int dir = pb != kt ? 0 : (reversed ? 1 : -1), side = dir * (4 * g - m);
    int soff[4];  // piece 4ks + g of row m (and of row 16 + m), ks = 0..3
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) soff[ks] = m * T::RS + 8 * wide_piece(m, 4 * ks + g);
    auto scores = [&](int buf) __attribute__((always_inline)) {
        if (w >= 3) return;
        f32x4 p0 = {0.f, 0.f, 0.f, 0.f}, p1 = p0;
        const u16 *keys = sB + buf * T::TILE + 16 * kt * T::RS, *pos = sA + buf * T::TILE + 16 * pb * T::RS;
#pragma unroll
        for (int ks = 0; ks < T::KS; ++ks) {
            const u32x4 a = *reinterpret_cast<const u32x4 *>(keys + soff[ks & 3] + 128 * (ks >> 2));
            const u32x4 b = *reinterpret_cast<const u32x4 *>(pos + soff[ks & 3] + 128 * (ks >> 2));
            if (ks & 1)
                p1 = TR::mfma(a, b, p1);
            else
                p0 = TR::mfma(a, b, p0);
        }
        p0 += p1;
#pragma unroll
        for (int q = 0; q < 4; ++q) p0[q] = side + dir * q >= 0 ? p0[q] : 0.f;
        uint32_t part[3][2];
        split3<Bf16>(p0[0], p0[1], part[0][0], part[1][0], part[2][0]);
        split3<Bf16>(p0[2], p0[3], part[0][1], part[1][1], part[2][1]);
#pragma unroll
        for (int x = 0; x < 3; ++x) sP[((buf * 3 + x) * 2 + pb) * 128 + 2 * l + kt] = u32x2{part[x][0], part[x][1]};
    };
    // output tile of chunk p, left in LDS by the compute wavefronts: one 16-byte piece per thread.  Unconditional like the
    // loads (see run_rounds): before the first tile and past the real columns the offset is out of range instead.
    auto store_out = [&](int p) __attribute__((always_inline)) {
        const u32x4 v = *reinterpret_cast<const u32x4 *>(sO + ((p - p0) & 1) * T::OTILE + crow * T::OS + ccol);
        const uint32_t off = (uint32_t)((first_row(p) + crow) * dj + ccol) * 2u;
        __builtin_amdgcn_raw_buffer_store_b128(v, rO, (int)(p >= p0 && c0 + ccol < dj ? off : kOobOffset), 0, 0);
    };
#pragma unroll
    for (int s = 0; s < PF; ++s) load_chunk(s, p0 + s);
    stage(0, 0);
    load_chunk(0, p0 + PF);
    __syncthreads();
    run_rounds<PF>(p0, p1, [&](int s, int p) __attribute__((always_inline)) {
        const int s1 = (s + 1) % PF, buf = s;  // (PF = 2: the LDS buffer is the register stage)
        stage(s1, buf ^ 1);
        load_chunk(s1, p + 1 + PF);
        if constexpr (!SUMS) {
            scores(buf);
            store_out(p - 2);
        }
        chunk_barrier();
    });
    if constexpr (!SUMS) {
        // the compute wavefronts finish the last chunk after the last barrier of the loop
        store_out(p1 - 2);
        chunk_barrier();
        store_out(p1 - 1);
    }
}

// Wavefront w of kWideCompute: state columns 16 (w & 3) .. + 15 of the slice, row half w >> 2.
// slots: those of this head and item; this group starts from the sum of slots first_slot .. grp (SUMS: slot grp + 1 receives
// the sum, or, with an empty range of chunks, slot 0 the start state).
template <class TR, int DI, bool SUMS>
__device__ __forceinline__ void wide_compute_role(const WideOp &op, int bh, int c0, const WideRange &rg, f32x4 *slots, int grp,
                                                  int first_slot, bool last_group, int w, int l, const u16 *sA, const u16 *sB,
                                                  const u16 *sC, u16 *sO, const u32x4 *sP, f32x4 *sX) {
    using T = WideTiling<DI>;
    constexpr bool FP16 = std::is_same<TR, Fp16>::value;
    constexpr int KS = T::KS / 2;
    const int g = l >> 4, m = l & 15;
    const int half = w >> 2, cw = 16 * (w & 3), i0 = half * (DI / 2);
    const int di = op.di, dj = op.dj, j = c0 + cw + m;  // this lane's state column
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    f32x4 S[2 * KS];
#pragma unroll
    for (int it = 0; it < 2 * KS; ++it) S[it] = zero;
    const int own = w * 2 * KS * 64 + l;
    const bool start = SUMS && rg.p0 == rg.p1;
    if ((!SUMS || start) && op.sin != nullptr && j < dj) {
        const float *src = op.sin + (size_t)bh * di * dj + j;
#pragma unroll
        for (int it = 0; it < 2 * KS; ++it)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int i = i0 + 32 * (it >> 1) + 8 * g + 4 * (it & 1) + q;
                if (i < di) S[it][q] = src[(size_t)i * dj];
            }
    }
    if (start) {
#pragma unroll
        for (int it = 0; it < 2 * KS; ++it) slots[own + 64 * it] = S[it];
        return;
    }
    if constexpr (!SUMS) {
        for (int gp = first_slot; gp <= grp; ++gp) {
            f32x4 t[2 * KS];
#pragma unroll
            for (int it = 0; it < 2 * KS; ++it) t[it] = slots[(size_t)gp * wide_slot_vectors(DI) + own + 64 * it];
#pragma unroll
            for (int it = 0; it < 2 * KS; ++it) S[it] += t[it];
        }
    }
    f32x4 o = zero;                // own part of A_c S_c, block `half` of the chunk whose scores are outstanding
    u32x4 cf = {0u, 0u, 0u, 0u};   // ... and its C fragment, keys in the order of the score operands
    int aoff[KS], boff[KS][2];  // A: piece 4ks + g of row m; B: rows 8g + m/4 (and + 4), piece 4ks + m%4, of this row half
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        const int c = i0 / 8 + 4 * ks, r = 8 * g + (m >> 2);
        aoff[ks] = m * T::RS + 8 * wide_piece(m, c + g);
        boff[ks][0] = r * T::RS + 8 * wide_piece(r, c + (m & 3));
        boff[ks][1] = (r + 4) * T::RS + 8 * wide_piece(r + 4, c + (m & 3));
    }
    auto finish = [&](int buf) __attribute__((always_inline)) {
        u32x4 ch = cf, cl = cf;
        if constexpr (FP16) fp16_as_bf16_pair(cf, ch, cl);
        u32x4 p[3];
#pragma unroll
        for (int x = 0; x < 3; ++x) p[x] = sP[((buf * 3 + x) * 2 + half) * 64 + l];
        const f32x4 other = sX[(buf * kWideCompute + (w ^ 4)) * 64 + l];
        const f32x4 hi = Bf16::mfma(ch, p[0], o + other);
        f32x4 rest = zero;
        if constexpr (FP16) {  // (the lo part of an infinite C is no number either: it stays out of `hi`)
            rest = Bf16::mfma(cl, p[2], rest);
            rest = Bf16::mfma(cl, p[1], rest);
            rest = Bf16::mfma(cl, p[0], rest);
        }
        rest = Bf16::mfma(ch, p[2], rest);
        rest = Bf16::mfma(ch, p[1], rest);
        f32x4 r = hi + rest;
        if (__any(any_nan(r))) r = number_or(r, hi);
        const u32x2 packed = {TR::pack2(r[0], r[1]), TR::pack2(r[2], r[3])};
        *reinterpret_cast<u32x2 *>(sO + buf * T::OTILE + (16 * half + m) * T::OS + cw + 4 * g) = packed;
    };
    __syncthreads();
    run_rounds<2>(rg.p0, rg.p1, [&](int buf, int p) __attribute__((always_inline)) {
        const u16 *tA = sA + buf * T::TILE, *tB = sB + buf * T::TILE, *tC = sC + buf * T::CTILE;
        if constexpr (!SUMS) {
            if (p > rg.p0) finish(buf ^ 1);
        }
        if constexpr (!SUMS) cf = cat(lds_col4(tC, T::CS, 4 * g, cw, m), lds_col4(tC, T::CS, 16 + 4 * g, cw, m));
        const u32x4 cu = cat(lds_col4(tC, T::CS, 8 * g, cw, m), lds_col4(tC, T::CS, 8 * g + 4, cw, m));
        float up = 1.f;
        f32x4 down = {1.f, 1.f, 1.f, 1.f};
        if constexpr (FP16 && !SUMS) {  // scale of this lane's half column: its largest entry to [2^14, 2^15)
            float mx = 0.f;
#pragma unroll
            for (int it = 0; it < 2 * KS; ++it)
#pragma unroll
                for (int q = 0; q < 4; ++q) mx = fmaxf(mx, __builtin_fabsf(S[it][q]));
            mx = fmaxf(mx, __shfl_xor(mx, 16));
            mx = fmaxf(mx, __shfl_xor(mx, 32));
            // exponent kept to where both the scale and its inverse are normal numbers, and every finite entry in range
            int e = (int)(bitcast<uint32_t>(mx) >> 23) - 127;
            e = e < -100 ? -100 : (e > 127 ? 127 : e);
            up = bitcast<float>((uint32_t)(127 + 14 - e) << 23);
#pragma unroll
            for (int q = 0; q < 4; ++q) down[q] = bitcast<float>((uint32_t)(127 - 14 + __shfl(e, 4 * g + q)) << 23);
        }
        f32x4 ah[2] = {zero, zero}, al[2] = {zero, zero};
        // One contraction step ahead: while the products of step ks are issued, the state rows of step ks + 1 are split and the
        // operands of that step are on their way from LDS (a matrix instruction and up to six vector ones in turn).
        u32x4 fa[2][2], fb[2][2], st[2][3];
        auto read = [&](int ks) __attribute__((always_inline)) {
#pragma unroll
            for (int x = 0; x < 2; ++x) {
                if constexpr (!SUMS) fa[ks & 1][x] = *reinterpret_cast<const u32x4 *>(tA + 16 * x * T::RS + aoff[ks]);
                // rows of state tile 2ks+x: columns 32ks + 8i + 4x .. +3 of B, i = 0..3
                fb[ks & 1][x] = cat(lds_read_tr16(tB + boff[ks][0] + 4 * x), lds_read_tr16(tB + boff[ks][1] + 4 * x));
            }
        };
        auto split = [&](int ks) __attribute__((always_inline)) {
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    uint32_t h, mid, lo;
                    split3<TR>(S[2 * ks + t][2 * q] * up, S[2 * ks + t][2 * q + 1] * up, h, mid, lo);
                    st[ks & 1][0][2 * t + q] = h;
                    st[ks & 1][1][2 * t + q] = mid;
                    st[ks & 1][2][2 * t + q] = lo;
                }
        };
        read(0);
        if constexpr (!SUMS) split(0);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            __builtin_amdgcn_sched_barrier(0);
            if (ks + 1 < KS) read(ks + 1);
            if constexpr (!SUMS) {
                if (ks + 1 < KS) split(ks + 1);
#pragma unroll
                for (int x = 2; x >= 0; --x)
#pragma unroll
                    for (int pb = 0; pb < 2; ++pb) {
                        f32x4 &acc = x == 0 ? ah[pb] : al[pb];
                        acc = TR::mfma(st[ks & 1][x], fa[ks & 1][pb], acc);
                    }
            }
#pragma unroll
            for (int t = 0; t < 2; ++t) S[2 * ks + t] = TR::mfma(fb[ks & 1][t], cu, S[2 * ks + t]);
            if constexpr (!SUMS) {
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x2, 6, 0);
                }
            }
        }
        if constexpr (!SUMS) {
#pragma unroll
            for (int pb = 0; pb < 2; ++pb) al[pb] += ah[pb];
            if (__any(any_nan(al[0]) | any_nan(al[1]))) {
                al[0] = number_or(al[0], ah[0]);
                al[1] = number_or(al[1], ah[1]);
            }
#pragma unroll
            for (int pb = 0; pb < 2; ++pb) {
                f32x4 r = al[pb];
                if constexpr (FP16) r *= down;
                if (pb == half)
                    o = r;
                else
                    sX[(buf * kWideCompute + w) * 64 + l] = r;
            }
        }
        chunk_barrier();
    });
    if constexpr (SUMS) {
#pragma unroll
        for (int it = 0; it < 2 * KS; ++it) slots[(size_t)(grp + 1) * wide_slot_vectors(DI) + own + 64 * it] = S[it];
        return;
    }
    finish((rg.p1 - 1 - rg.p0) & 1);
    chunk_barrier();
    if (op.sout != nullptr && last_group && j < dj) {
        float *dst = op.sout + (size_t)bh * di * dj + j;
#pragma unroll
        for (int it = 0; it < 2 * KS; ++it)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int i = i0 + 32 * (it >> 1) + 8 * g + 4 * (it & 1) + q;
                if (i < di) dst[(size_t)i * dj] = S[it][q];
            }
    }
}

// 768 threads: wavefronts 0..7 compute, 8..11 load.  Grid: grid_for(BH, set.items, groups, set.xcds), groups = G, or for the sums
// G - first_slot, so that the slices and ops of a head and group run on one XCD and share its tiles through that L2.
template <class TR, int DI, bool SUMS>
__global__ __launch_bounds__(64 * (kWideCompute + kWideLoad)) void wide_scan_kernel(WideSet set, int BH, int N, int nchunks) {
    using T = WideTiling<DI>;
    __shared__ __attribute__((aligned(16))) unsigned char wide_smem[T::LDS];
    u16 *sA = reinterpret_cast<u16 *>(wide_smem);
    u16 *sB = sA + 2 * T::TILE, *sC = sB + 2 * T::TILE, *sO = sC + 2 * T::CTILE;
    u32x4 *sP = reinterpret_cast<u32x4 *>(sO + 2 * T::OTILE);
    f32x4 *sX = reinterpret_cast<f32x4 *>(sP + T::SCORES);
    const WorkItem wi = decode_workgroup(set.items, BH, set.xcds);
    if (wi.grp >= (SUMS ? set.G - set.first_slot : set.G)) return;
    const bool start = SUMS && wi.grp == set.G - 1;  // this workgroup only puts the start state into slot 0
    int which = 0, slice = wi.prob;
    while (which + 1 < set.count && slice >= set.op[which].slices) slice -= set.op[which++].slices;
    const WideOp &op = set.op[which];
    const WideRange rg = {N, nchunks, start ? 0 : wi.grp * set.cpg, start ? 0 : min((wi.grp + 1) * set.cpg, nchunks)};
    f32x4 *slots = set.slots + ((size_t)wi.bh * set.items + wi.prob) * set.G * wide_slot_vectors(DI);
    const int tid = threadIdx.x;
    if constexpr (!SUMS) {  // the score tiles on the other side of the diagonal are never written: zero
        for (int x = tid; x < T::SCORES; x += 64 * (kWideCompute + kWideLoad)) sP[x] = u32x4{0u, 0u, 0u, 0u};
        __syncthreads();
    }
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    if (w < kWideCompute)
        wide_compute_role<TR, DI, SUMS>(op, wi.bh, slice * kWideSlice, rg, slots, wi.grp, set.first_slot, wi.grp == set.G - 1, w,
                                        tid & 63, sA, sB, sC, sO, sP, sX);
    else if (!start)
        wide_loader_role<TR, DI, SUMS>(op, wi.bh, slice * kWideSlice, rg, tid - 64 * kWideCompute, sA, sB, sC, sO,
                                       reinterpret_cast<u32x2 *>(sP));
}

}  // namespace cott
