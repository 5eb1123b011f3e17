// Launches of the wide-head scan.
#include "cott_wide.h"
#include "cott_launch.h"
#include "../../include/cottention.h"

namespace cott {
namespace {

int wide_pad(int di) { return di <= 128 ? 128 : (di <= 192 ? 192 : 256); }

// Groups a sequence is cut into: as many as keep the launch at one workgroup per CU (the (head, group) units are dealt round
// the XCDs, and the fullest XCD has to hold its units' workgroups at once), of eight chunks at least, at most 16 (a group
// reads the slots of all groups before it).  Sequences below 24 chunks stay whole (2 heads N512 D256, forward 28 us; two
// launches of a few us each would have to save more).  Whole / groups, us: forward 16 heads D256 N768 40.8 / 27.4, N1024
// 53.1 / 30.6, N4096 194 / 95; 2 heads N4096 190 / 39, N16384 760 / 83; gradients 2 heads N1024 54 / 30, N4096 197 / 52.  More
// groups than an XCD holds at once are slower (gradients of 2 heads N4096, with the two-term splits: 10 groups 67 us, 8
// groups 47).
int wide_groups(long BH, int items, int nchunks, int cus, int xcds) {
    if (nchunks < 24) return 1;
    long g = cus / xcds / items * xcds / BH;
    if (g > nchunks / 8) g = nchunks / 8;
    if (g > 16) g = 16;
    if (g < 2) return 1;
    const int cpg = (int)((nchunks + g - 1) / g);
    return (nchunks + cpg - 1) / cpg;
}

int wide_chunks(int N) { return (N + kWideChunk - 1) / kWideChunk; }

// Slots of one launch in G > 1 groups: BH heads, `items` slices, the start state and all groups but the last.
size_t wide_slot_bytes(long BH, int items, int G, int pad) {
    return G > 1 ? (size_t)BH * items * G * wide_slot_vectors(pad) * sizeof(f32x4) : 0;
}

template <class TR, int DI>
hipError_t launch_set(WideSet set, int BH, int N, hipStream_t stream) {
    const int nchunks = wide_chunks(N);
    const dim3 block(64 * (kWideCompute + kWideLoad));
    set.first_slot = 1;
    if (set.G > 1) {
        for (const WideOp &o : set.op)
            if (o.sin != nullptr) set.first_slot = 0;
        ProfScope ps(K_WIDE_SUMS, stream);
        wide_scan_kernel<TR, DI, true><<<dim3(grid_for(BH, set.items, set.G - set.first_slot, set.xcds)), block, 0, stream>>>(
            set, BH, N, nchunks);
        for (WideOp &o : set.op) o.sin = nullptr;
    }
    ProfScope ps(K_WIDE_SCAN, stream);
    // A launch holds fewer than 2^32 threads: more heads than that (whole sequences, then) take several launches.
    const long most = ((1L << 32) - 1) / (block.x * (long)set.items) / set.G - set.xcds;
    const int step = set.G > 1 || BH <= most ? BH : (int)most;
    for (int bh = 0; bh < BH; bh += step) {
        const int heads = BH - bh < step ? BH - bh : step;
        WideSet part = set;
        for (int i = 0; i < set.count; ++i) {
            WideOp &o = part.op[i];
            const size_t rows = (size_t)bh * N, state = (size_t)bh * o.di * o.dj;
            o.A += rows * o.di;
            o.B += rows * o.di;
            o.C += rows * o.dj;
            o.O += rows * o.dj;
            if (o.sin != nullptr) o.sin += state;
            if (o.sout != nullptr) o.sout += state;
        }
        wide_scan_kernel<TR, DI, false><<<dim3(grid_for(heads, set.items, set.G, set.xcds)), block, 0, stream>>>(part, heads, N, nchunks);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

template <class TR>
hipError_t launch_typed(const OpDesc *ops, int n, int BH, int N, int cus, int xcds, char *ws, size_t ws_bytes,
                        hipStream_t stream) {
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
        const int nchunks = wide_chunks(N);
        set.G = wide_groups(BH, set.items, nchunks, cus, xcds);
        const size_t need = wide_slot_bytes(BH, set.items, set.G, pad);
        // These widths needed no workspace on the plain-FMA kernel, so calls without one stay accepted: sequences are then
        // walked whole, the sums in another order (results equal to rounding, not bit for bit) and with few heads slower.
        if (need > ws_bytes) set.G = 1;
        set.cpg = (nchunks + set.G - 1) / set.G;
        if (set.G > 1) {
            set.slots = reinterpret_cast<f32x4 *>(ws);
            ws += need;
            ws_bytes -= need;
        }
        const hipError_t e = pad == 128   ? launch_set<TR, 128>(set, BH, N, stream)
                             : pad == 192 ? launch_set<TR, 192>(set, BH, N, stream)
                                          : launch_set<TR, 256>(set, BH, N, stream);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace

size_t wide_workspace(const int *di, const int *dj, int n, long BH, int N, int cus, int xcds) {
    size_t total = 0;
    for (int pad = 128; pad <= 256; pad += 64) {
        int items = 0;
        for (int i = 0; i < n; ++i)
            if (wide_pad(di[i]) == pad) items += (dj[i] + kWideSlice - 1) / kWideSlice;
        if (items > 0) total += wide_slot_bytes(BH, items, wide_groups(BH, items, wide_chunks(N), cus, xcds), pad);
    }
    return total;
}

hipError_t launch_wide(int dtype, const OpDesc *ops, int n, int BH, int N, int cus, int xcds, void *ws, size_t ws_bytes,
                       hipStream_t stream) {
    char *w = static_cast<char *>(ws);
    if (dtype == COTT_BF16) return launch_typed<Bf16>(ops, n, BH, N, cus, xcds, w, ws_bytes, stream);
    if (dtype == COTT_F16) return launch_typed<Fp16>(ops, n, BH, N, cus, xcds, w, ws_bytes, stream);
    return hipErrorInvalidValue;
}

}  // namespace cott
