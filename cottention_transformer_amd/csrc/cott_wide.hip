// Launches of the wide-head scan.
#include "cott_wide.h"
#include "cott_launch.h"
#include "../../include/cottention.h"

namespace cott {
namespace {

int wide_pad(int di) { return di <= 128 ? 128 : (di <= 192 ? 192 : 256); }

template <class TR, int DI>
hipError_t launch_set(const WideSet &set, int BH, int N, int prof_id, hipStream_t stream) {
    ProfScope ps(prof_id, stream);
    const int nchunks = (N + kWideChunk - 1) / kWideChunk;
    wide_scan_kernel<TR, DI><<<dim3(grid_for(BH, set.items, 1, set.xcds)), dim3(64 * (kWideCompute + kWideLoad)), 0, stream>>>(set, BH, N, nchunks);
    return hipGetLastError();
}

template <class TR>
hipError_t launch_typed(const OpDesc *ops, int n, int BH, int N, int xcds, int prof_id, hipStream_t stream) {
    // one launch per padded width of the contracted dim (the gradients of square heads are one)
    for (int pad = 128; pad <= 256; pad += 64) {
        WideSet set{};
        set.xcds = xcds;
        for (int i = 0; i < n; ++i) {
            const OpDesc &o = ops[i];
            if (wide_pad(o.di) != pad) continue;
            WideOp &w = set.op[set.count++];
            w.A = static_cast<const u16 *>(o.A);
            w.B = static_cast<const u16 *>(o.B);
            w.C = static_cast<const u16 *>(o.C);
            w.O = static_cast<u16 *>(o.O);
            w.sin = static_cast<const float *>(o.sin);
            w.sout = static_cast<float *>(o.sout);
            w.di = o.di;
            w.dj = o.dj;
            w.reversed = o.reversed;
            w.slices = (o.dj + kWideSlice - 1) / kWideSlice;
            set.items += w.slices;
        }
        if (set.count == 0) continue;
        const hipError_t e = pad == 128   ? launch_set<TR, 128>(set, BH, N, prof_id, stream)
                             : pad == 192 ? launch_set<TR, 192>(set, BH, N, prof_id, stream)
                                          : launch_set<TR, 256>(set, BH, N, prof_id, stream);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace

hipError_t launch_wide(int dtype, const OpDesc *ops, int n, int BH, int N, int xcds, int prof_id, hipStream_t stream) {
    if (dtype == COTT_BF16) return launch_typed<Bf16>(ops, n, BH, N, xcds, prof_id, stream);
    if (dtype == COTT_F16) return launch_typed<Fp16>(ops, n, BH, N, xcds, prof_id, stream);
    return hipErrorInvalidValue;
}

}  // namespace cott
