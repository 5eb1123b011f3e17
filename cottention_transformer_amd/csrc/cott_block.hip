// The small passes of an attention block around its GEMMs: conversions of hidden states and weights, the keep mask and its
// counts, sums of gradients over rows.  Each replaces several elementwise or reduction launches of a few us; in a block's
// step both the device time and the launches themselves count (a launch costs 5 to 10 us of host time, and the step is close
// to host-bound).
#include "cott_common.h"
#include "cott_launch.h"
#include "../../include/cottention.h"

namespace cott {
namespace {

constexpr int kBlock = 256;

struct ConvertArgs {
    const float *src[COTT_CONVERT_MAX];
    u16 *dst[COTT_CONVERT_MAX];
    long n[COTT_CONVERT_MAX];
    long first[COTT_CONVERT_MAX + 1];  // first piece of 8 elements of each array in the grid's numbering
    int count;
};

// fp32 -> 16 bits, rounded to nearest even; a piece of eight elements per thread (two 16-byte loads, one 16-byte store).
// Bound by memory: 16384 x 1024 hidden states and three 1024 x 1024 weights (119 MB moved) in one launch 23.5 us, where four
// launches of a general elementwise kernel took 30.
template <class TR>
__global__ __launch_bounds__(kBlock) void convert_kernel(ConvertArgs a) {
    const long piece = (long)blockIdx.x * kBlock + threadIdx.x;
    if (piece >= a.first[a.count]) return;
    int which = 0;
#pragma unroll
    for (int i = 1; i < COTT_CONVERT_MAX; ++i) which += i < a.count && piece >= a.first[i];
    const long at = 8 * (piece - a.first[which]);
    const float *src = a.src[which] + at;
    u16 *dst = a.dst[which] + at;
    const long left = a.n[which] - at;
    if (left >= 8) {
        const f32x4 x = reinterpret_cast<const f32x4 *>(src)[0], y = reinterpret_cast<const f32x4 *>(src)[1];
        *reinterpret_cast<u32x4 *>(dst) = u32x4{TR::pack2(x[0], x[1]), TR::pack2(x[2], x[3]), TR::pack2(y[0], y[1]), TR::pack2(y[2], y[3])};
    } else {
        for (long i = 0; i < left; ++i) dst[i] = TR::from_float(src[i]);
    }
}

template <class E>
__device__ __forceinline__ bool is_zero(E x) {
    return x == (E)0;  // (not so for a NaN)
}
template <>
__device__ __forceinline__ bool is_zero<u16>(u16 x) {  // bf16 and fp16 alike: +0 and -0
    return (x & 0x7fffu) == 0;
}

// One workgroup of 16 wavefronts per batch element walks the positions in tiles of 8192, eight consecutive ones per thread.
// RUNNING: cnt[s] = kept positions up to and with s, else their number in the whole sequence.  The counts inside a thread and
// a wavefront come from bit counts of ballots; one exchange through LDS per tile.  8 x 2048: 4.9 us, where the comparison,
// the conversion to numbers and the cumulative sum took 23 in three launches.  Bound by the one workgroup's walk, 1 us per 1000
// positions: callers with a few long sequences do better with a reduction over the whole chip (ops.keep_and_counts_preferred).
template <class E, bool RUNNING>
__global__ __launch_bounds__(1024) void keep_counts_kernel(const E *mask, unsigned char *keep, float *cnt, int N) {
    __shared__ int totals[16];
    const int tid = threadIdx.x, l = tid & 63, w = tid >> 6;
    mask += (size_t)blockIdx.x * N;
    keep += (size_t)blockIdx.x * N;
    cnt += (size_t)blockIdx.x * N;
    int before = 0;  // kept in the tiles before this one
    for (int base = 0; base < N; base += 8192) {
        const int s0 = base + 8 * tid;
        uint32_t bits = 0;
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (s0 + i < N && is_zero<E>(mask[s0 + i])) bits |= 1u << i;
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (s0 + i < N) keep[s0 + i] = (bits >> i) & 1u;
        const int own = __builtin_popcount(bits);
        int upto = own;  // inclusive sum over the lanes of the wavefront
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int from = __shfl_up(upto, off, 64);
            if (l >= off) upto += from;
        }
        if (l == 63) totals[w] = upto;
        __syncthreads();
        int all = 0, waves_before = 0;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            waves_before += i < w ? totals[i] : 0;
            all += totals[i];
        }
        if (RUNNING) {
            int c = before + waves_before + upto - own;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                c += (bits >> i) & 1u;
                if (s0 + i < N) cnt[s0 + i] = (float)c;
            }
        }
        before += all;
        __syncthreads();
    }
    if (!RUNNING)
        for (int s = tid; s < N; s += 1024) cnt[s] = (float)before;
}

// Sum of v over the workgroup, in every thread of the first wavefront.
__device__ __forceinline__ float block_sum(float v, float *part) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
    __syncthreads();
    v = threadIdx.x < 16 ? part[threadIdx.x] : 0.f;
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// out[h] = sum over b and s of rows[b][h][s]: one workgroup per head, eight loads in flight per thread whatever the split into b
// and s (a loop over b with one load each took 10 us at 32 x 12 x 512).  5.6 us there and at 8 x 16 x 2048, where a general
// reduction takes 10.4 and 11.0.  Bound by the one workgroup, 20 us per 100000 rows: ops.head_sums adds longer ones in two steps.
__global__ __launch_bounds__(1024) void head_sums_kernel(const float *rows, float *out, int B, int H, int N) {
    __shared__ float part[16];
    const float *head = rows + (size_t)blockIdx.x * N;
    const size_t step = (size_t)H * N;
    const long total = (long)B * N;
    float sum = 0.f;
    for (long base = threadIdx.x; base < total; base += 8 * 1024) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const long i = base + 1024 * u;
            const uint32_t b = (uint32_t)(i < total ? i : 0) / (uint32_t)N;  // (at most 2^32 rows of a head: see launch_head_sums)
            v[u] = i < total ? head[b * step + (size_t)(i - (long)b * N)] : 0.f;
        }
        sum += ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
    }
    sum = block_sum(sum, part);
    if (threadIdx.x == 0) out[blockIdx.x] = sum;
}

// Partial column sums of a 16-bit (rows, cols) matrix: workgroup (x, y) adds the rows of share y for 256 columns, eight
// columns per thread in 32 lanes, eight rows side by side, and leaves part[y][col].  Unrolled by four: 64 bytes in flight per
// thread.  Bound by memory: 16384 x 2304 (75 MB) 12.4 us and 3.9 for the parts, where a general reduction and its two memsets
// take 37.
template <class TR>
__global__ __launch_bounds__(kBlock) void column_sums_kernel(const u16 *x, float *part, long rows, int cols, long ld, long share) {
    __shared__ float tile[8][256 + 8];
    const int lane = threadIdx.x % 32, sub = threadIdx.x / 32, col = 256 * blockIdx.x + 8 * lane;
    const long r0 = blockIdx.y * share, r1 = r0 + share < rows ? r0 + share : rows;
    float sum[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (col < cols) {
#pragma unroll 4
        for (long r = r0 + sub; r < r1; r += 8) {
            const u32x4 v = *reinterpret_cast<const u32x4 *>(x + r * ld + col);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                sum[2 * i] += TR::to_float((u16)(v[i] & 0xffffu));
                sum[2 * i + 1] += TR::to_float((u16)(v[i] >> 16));
            }
        }
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) tile[sub][8 * lane + i] = sum[i];
    __syncthreads();
    const int c = threadIdx.x;
    if (256 * (int)blockIdx.x + c < cols) {
        float s = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) s += tile[i][c];
        part[(size_t)blockIdx.y * cols + 256 * blockIdx.x + c] = s;
    }
}
// Where consecutive blocks of one row of sums go: each into an array of its own (gradients of several parameters).
struct Blocks {
    float *out[COTT_CONVERT_MAX];
    long first[COTT_CONVERT_MAX + 1];  // first element of each block, and their total
    int count;
    __device__ __forceinline__ float *at(long e) const {
        int which = 0;
#pragma unroll
        for (int i = 1; i < COTT_CONVERT_MAX; ++i) which += i < count && e >= first[i];
        return out[which] + (e - first[which]);
    }
};

// Sum over the parts of every column: 32 columns per workgroup, eight threads to a column.
__global__ __launch_bounds__(kBlock) void add_parts_kernel(const float *part, Blocks to, int cols, int parts) {
    __shared__ float tile[8][32];
    const int c = threadIdx.x % 32, sub = threadIdx.x / 32, col = 32 * blockIdx.x + c;
    float s = 0.f;
    if (col < cols) {
#pragma unroll 8
        for (int p = sub; p < parts; p += 8) s += part[(size_t)p * cols + col];
    }
    tile[sub][c] = s;
    __syncthreads();
    if (threadIdx.x < 32 && col < cols) {
        s = tile[0][c];
#pragma unroll
        for (int i = 1; i < 8; ++i) s += tile[i][c];
        *to.at(col) = s;
    }
}

// Sum over the pieces of a weight gradient, (pieces, total) fp32: four elements per thread.  Bound by memory: 4 pieces of three 1024 x
// 1024 weights (63 MB) 10.9 us, 8 of three 768 x 768 (64 MB) 11.8; a general reduction for every weight 24 and 21.
__global__ __launch_bounds__(kBlock) void add_pieces_kernel(const float *parts, Blocks to, int pieces) {
    const long e = 4 * ((long)blockIdx.x * kBlock + threadIdx.x), total = to.first[to.count];
    if (e >= total) return;
    f32x4 sum = *reinterpret_cast<const f32x4 *>(parts + e);
#pragma unroll 4
    for (int p = 1; p < pieces; ++p) sum += *reinterpret_cast<const f32x4 *>(parts + p * total + e);
    *reinterpret_cast<f32x4 *>(to.at(e)) = sum;
}

Blocks blocks_of(float *const *out, const long *n, int count) {
    Blocks b{};
    b.count = count;
    for (int i = 0; i < count; ++i) {
        b.out[i] = out[i];
        b.first[i + 1] = b.first[i] + n[i];
    }
    return b;
}

}  // namespace

hipError_t launch_convert(int dtype, const float *const *src, void *const *dst, const long *n, int count, hipStream_t stream) {
    ConvertArgs a{};
    a.count = count;
    for (int i = 0; i < count; ++i) {
        a.src[i] = src[i];
        a.dst[i] = static_cast<u16 *>(dst[i]);
        a.n[i] = n[i];
        a.first[i + 1] = a.first[i] + (n[i] + 7) / 8;
    }
    const long blocks = (a.first[count] + kBlock - 1) / kBlock;
    if (blocks == 0) return hipSuccess;
    if (blocks > 0x7fffffL) return hipErrorInvalidValue;  // (2^31 threads)
    ProfScope prof(K_PREP, stream);
    if (dtype == COTT_BF16)
        convert_kernel<Bf16><<<dim3((unsigned)blocks), dim3(kBlock), 0, stream>>>(a);
    else
        convert_kernel<Fp16><<<dim3((unsigned)blocks), dim3(kBlock), 0, stream>>>(a);
    return hipGetLastError();
}

hipError_t launch_keep_counts(const void *mask, int bytes, unsigned char *keep, float *cnt, int B, int N, bool running,
                              hipStream_t stream) {
    ProfScope prof(K_PREP, stream);
    const dim3 grid(B), block(1024);
    if (bytes == 4) {
        const float *m = static_cast<const float *>(mask);
        if (running)
            keep_counts_kernel<float, true><<<grid, block, 0, stream>>>(m, keep, cnt, N);
        else
            keep_counts_kernel<float, false><<<grid, block, 0, stream>>>(m, keep, cnt, N);
    } else {
        const u16 *m = static_cast<const u16 *>(mask);
        if (running)
            keep_counts_kernel<u16, true><<<grid, block, 0, stream>>>(m, keep, cnt, N);
        else
            keep_counts_kernel<u16, false><<<grid, block, 0, stream>>>(m, keep, cnt, N);
    }
    return hipGetLastError();
}

hipError_t launch_head_sums(const float *rows, float *out, int B, int H, int N, hipStream_t stream) {
    if ((long)B * N >= (1L << 32)) return hipErrorInvalidValue;
    ProfScope prof(K_PREP, stream);
    head_sums_kernel<<<dim3(H), dim3(1024), 0, stream>>>(rows, out, B, H, N);
    return hipGetLastError();
}

// Shares of at least 64 rows, as many as give four workgroups to a CU: enough bytes in flight for the memory's rate.
int column_sum_parts(long rows, int cols, int cus) {
    const long wide = (cols + 255) / 256;
    long parts = 4L * cus / wide;
    if (parts > rows / 64) parts = rows / 64;
    return (int)(parts < 1 ? 1 : parts);
}

hipError_t launch_column_sums(int dtype, const void *x, float *const *out, const long *n, int count, long rows, int cols, long ld,
                              int parts, float *ws, hipStream_t stream) {
    ProfScope prof(K_PREP, stream);
    const long share = (rows + parts - 1) / parts;
    const u16 *src = static_cast<const u16 *>(x);
    auto sums = [&](const u16 *from, float *to, int width) {
        const dim3 grid((width + 255) / 256, parts), block(kBlock);
        if (dtype == COTT_BF16)
            column_sums_kernel<Bf16><<<grid, block, 0, stream>>>(from, to, rows, width, ld, share);
        else
            column_sums_kernel<Fp16><<<grid, block, 0, stream>>>(from, to, rows, width, ld, share);
    };
    if (parts > 1) {
        sums(src, ws, cols);
        add_parts_kernel<<<dim3((cols + 31) / 32), dim3(kBlock), 0, stream>>>(ws, blocks_of(out, n, count), cols, parts);
    } else {  // few rows: every block by itself
        long first = 0;
        for (int i = 0; i < count; first += n[i++])
            if (n[i] > 0) sums(src + first, out[i], (int)n[i]);
    }
    return hipGetLastError();
}

hipError_t launch_add_pieces(const float *parts, float *const *out, const long *n, int count, int pieces, hipStream_t stream) {
    const Blocks to = blocks_of(out, n, count);
    const long blocks = (to.first[count] / 4 + kBlock - 1) / kBlock;
    if (blocks == 0) return hipSuccess;
    if (blocks > 0x7fffffL) return hipErrorInvalidValue;  // (2^31 threads)
    ProfScope prof(K_PREP, stream);
    add_pieces_kernel<<<dim3((unsigned)blocks), dim3(kBlock), 0, stream>>>(parts, to, pieces);
    return hipGetLastError();
}

}  // namespace cott
