// Projections of the one new token of a decode step (x w^T for at most 16 rows of x).
//
// Bound: the weights, read once (E = 2048, bf16: 8.4 MB a matrix, which stays in the last-level cache from token to
// token).  A workgroup of eight wavefronts owns 16 output columns and cuts the contraction in eight, so that a wavefront
// has its whole share (E = 2048: eight 16-byte loads a lane) in flight at once and q, k and v together are 384
// workgroups.  The rows of x are the second matrix operand, padded to 16 with zeros by the buffer's range check: up to
// 16 sequences cost what one does.  Contiguous steps per wavefront: two neighbouring 64-byte halves of a line are
// fetched by the same wavefront, one after the other.  E = 2048, one row: q, k and v in one launch and the output
// projection 6.2 us on average, where the GEMM library takes four launches of 8.1 us and 25 us of host time each.
#include "cott_common.h"
#include "cott_launch.h"
#include "../../include/cottention.h"

namespace cott {
namespace {

constexpr int kTokenWaves = 8;
struct TokenLinear {
    const u16 *x;     // (rows, in)
    const u16 *w[3];  // (out, in) each
    u16 *y[3];        // (rows, out) each
    int rows, in, out;
};

template <class TR>
__global__ __launch_bounds__(64 * kTokenWaves) void token_linear_kernel(TokenLinear a) {
    constexpr int U = 8;
    __shared__ f32x4 part[kTokenWaves * 64];
    const int tid = threadIdx.x, l = tid & 63, g = l >> 4, m = l & 15;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tiles = a.out / 16, mat = blockIdx.x / tiles, o0 = (blockIdx.x % tiles) * 16;
    const rsrc_t rx = make_rsrc(a.x, (uint32_t)a.rows * a.in * 2u);
    const rsrc_t rw = make_rsrc(a.w[mat] + (size_t)o0 * a.in, 16u * a.in * 2u);
    const int steps = a.in / 32, per = (steps + kTokenWaves - 1) / kTokenWaves;
    const int s1 = min((w + 1) * per, steps);
    const uint32_t row = (uint32_t)(m * a.in + 8 * g) * 2u;
    f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    for (int s0 = w * per; s0 < s1; s0 += U) {
        u32x4 wf[U], xf[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t off = s0 + u < s1 ? row + (uint32_t)(s0 + u) * 64u : kOobOffset;
            wf[u] = buf_load16(rw, off);
            xf[u] = buf_load16(rx, off);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) acc[u & 1] = TR::mfma(wf[u], xf[u], acc[u & 1]);
    }
    part[tid] = acc[0] + acc[1];
    __syncthreads();
    if (tid < 64 && m < a.rows) {  // lane: output columns o0 + 4g .. + 3 of row m
        f32x4 y = part[l];
#pragma unroll
        for (int i = 1; i < kTokenWaves; ++i) y += part[64 * i + l];
        const u32x2 v = {TR::pack2(y[0], y[1]), TR::pack2(y[2], y[3])};
        *reinterpret_cast<u32x2 *>(a.y[mat] + (size_t)m * a.out + o0 + 4 * g) = v;
    }
}

}  // namespace

hipError_t launch_token_linear(int dtype, const void *x, const void *const w[3], void *const y[3], int count, int rows, int in,
                               int out, hipStream_t stream) {
    TokenLinear a{};
    a.x = static_cast<const u16 *>(x);
    for (int i = 0; i < count; ++i) {
        a.w[i] = static_cast<const u16 *>(w[i]);
        a.y[i] = static_cast<u16 *>(y[i]);
    }
    a.rows = rows;
    a.in = in;
    a.out = out;
    ProfScope ps(K_TOKEN_LINEAR, stream);
    const dim3 grid((unsigned)(count * (out / 16))), block(64 * kTokenWaves);
    if (dtype == COTT_BF16)
        token_linear_kernel<Bf16><<<grid, block, 0, stream>>>(a);
    else if (dtype == COTT_F16)
        token_linear_kernel<Fp16><<<grid, block, 0, stream>>>(a);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

}  // namespace cott
