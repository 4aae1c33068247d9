// solve.hip -- control-point solve kernels and launchers (the device code
// is in solve_impl.hpp).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "solve_impl.hpp"

namespace intp_amd {

namespace {

constexpr int kMaxTileThreads = 512;
// LDS of a tiled workgroup: two workgroups per CU on gfx950 (160 KB).
constexpr int64_t kTileLdsBudget = 80 * 1024;

template <int BW, bool CYC, typename T, typename C, int B>
__global__ __launch_bounds__(kSolveBlock) void solve_kernel(SolveParams sp) {
    const int64_t line = static_cast<int64_t>(blockIdx.x) * kSolveBlock + threadIdx.x;
    warm_factors<BW, CYC, C, kSolveBlock>(sp, sp.n);  // a few lines: all in block 0
    if (line >= sp.nlines) return;
    const int64_t o = line / sp.inner, ii = line - o * sp.inner;
    substitute<BW, CYC, C, T, B>(static_cast<T*>(sp.x) + o * sp.n * sp.inner + ii, sp.inner, sp.n, sp);
}

// Waves per SIMD the tile kernel is built for: three (168 VGPRs) where that
// does not spill, so that tiles of short lines share a CU three at a time
// (150^3 cubic, one axis: 34 us at two, 27 us at three; four spill).
template <int BW, bool CYC, typename C>
constexpr int tile_waves() {
    return !CYC && (sizeof(C) == 4 || BW <= 2) ? 3 : 2;
}

template <int BW, bool CYC, typename T, typename C>
__global__ __launch_bounds__(kMaxTileThreads, (tile_waves<BW, CYC, C>())) void solve_tile_kernel(SolveParams sp) {
    extern __shared__ __align__(16) unsigned char tile_bytes[];
    __shared__ int64_t dst_base[kMaxTileLines];
    __shared__ int64_t src_base[kMaxTileLines];
    const int nt = static_cast<int>(blockDim.x);  // a power of two
    solve_tile<BW, CYC, T, C>(sp, static_cast<int64_t>(blockIdx.x) * sp.lines_per_block, tile_bytes, dst_base,
                              src_base, static_cast<int>(threadIdx.x + 64 * blockIdx.x) & (nt - 1), nt);
}

template <int BW, bool CYC, typename T, typename C>
hipError_t launch_lines(const SolveParams& p, int threads, hipStream_t s) {
    if (p.lines_per_block > 0) {
        const int lpb = p.lines_per_block;
        const int64_t blocks = (p.nlines + lpb - 1) / lpb;
        if (blocks > 0x7FFFFFFF) return hipErrorInvalidValue;
        const size_t lds = static_cast<size_t>(tile_elements(p.n, lpb, p.inner) + edge_elements(p.n, BW, p)) * sizeof(C);
        hipLaunchKernelGGL((solve_tile_kernel<BW, CYC, T, C>), dim3(static_cast<unsigned>(blocks)),
                           dim3(static_cast<unsigned>(threads)), lds, s, p);
        return hipGetLastError();
    }
    const int64_t blocks = (p.nlines + kSolveBlock - 1) / kSolveBlock;
    hipLaunchKernelGGL((solve_kernel<BW, CYC, T, C, batch_rows<BW, CYC>()>), dim3(static_cast<unsigned>(blocks)),
                       dim3(kSolveBlock), 0, s, p);
    return hipGetLastError();
}

template <typename T>
__global__ __launch_bounds__(kSolveBlock) void shift_copy_kernel(ShiftParams sp) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kSolveBlock + threadIdx.x;
    if (i >= sp.total) return;
    int64_t rem = i, dst = 0, mul = 1;
    for (int d = sp.dim - 1; d >= 0; --d) {
        const int64_t n = sp.n[d];
        const int64_t id = rem % n;
        rem /= n;
        int64_t w = id + sp.shift[d];
        if (w >= n) w -= n;
        dst += w * mul;
        mul *= n;
    }
    static_cast<T*>(sp.dst)[dst] = static_cast<T>(sp.src[i]);
}

template <int BW, typename T, typename C>
hipError_t launch_bw(bool cyclic, const SolveParams& p, int threads, hipStream_t s) {
    if (p.nlines == 0) return hipSuccess;
    if (p.lines_per_block > 0) {
        // whole lanes per line, every segment's lane present, rows in 32 bits
        const int lpb = p.lines_per_block;
        if (lpb > kMaxTileLines || threads > kMaxTileThreads || threads % lpb != 0 || threads % 64 != 0 ||
            (threads & (threads - 1)) != 0 ||
            (lpb & (lpb - 1)) != 0 || p.segs < 0 || p.segs > threads / lpb || (p.segs > 1 && p.segs < BW) || threads / lpb < BW ||
            p.n >= (int64_t{1} << 24))
            return hipErrorInvalidValue;
    } else if (p.src || p.accum) {
        return hipErrorInvalidValue;  // the HBM kernel solves in place only
    }
    if (!cyclic) return launch_lines<BW, false, T, C>(p, threads, s);
    // a periodic order k has band width k / 2
    if constexpr (2 * BW <= kMaxOrder) return launch_lines<BW, true, T, C>(p, threads, s);
    return hipErrorNotSupported;
}

template <typename T, typename C>
hipError_t launch_typed(int bw, bool cyclic, const SolveParams& p, int threads, hipStream_t s) {
    switch (bw) {
        case 0: return launch_bw<0, T, C>(cyclic, p, threads, s);
        case 1: return launch_bw<1, T, C>(cyclic, p, threads, s);
        case 2: return launch_bw<2, T, C>(cyclic, p, threads, s);
        case 3: return launch_bw<3, T, C>(cyclic, p, threads, s);
        case 4: return launch_bw<4, T, C>(cyclic, p, threads, s);
        case 5: return launch_bw<5, T, C>(cyclic, p, threads, s);
        case 6: return launch_bw<6, T, C>(cyclic, p, threads, s);
        default: return hipErrorNotSupported;
    }
}

}  // namespace

hipError_t launch_solve(int bw, bool cyclic, SolveTypes types, const SolveParams& p, int threads, hipStream_t s) {
    switch (types) {
        case SolveTypes::kF64: return launch_typed<double, double>(bw, cyclic, p, threads, s);
        case SolveTypes::kF32: return launch_typed<float, float>(bw, cyclic, p, threads, s);
        case SolveTypes::kF32StoreF64Compute: return launch_typed<float, double>(bw, cyclic, p, threads, s);
        default: return hipErrorInvalidValue;
    }
}

TilePlan solve_tile_plan(const SolveParams& p, int bw, bool cyclic, int compute_bytes) {
    TilePlan plan;
    int dev = 0, max_lds = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&max_lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess)
        return plan;
    const int64_t n = p.n, inner = p.inner;
    // lines long enough for rows of equal factors (and, cyclic, for the
    // strips' prefix) to matter; shorter ones are substituted plainly
    // (one axis, one segment against plain: n = 97, order 4 20.6 / 17.8 us;
    // n = 150, order 3 28 / 29 us)
    SolveParams cut = p;
    cut.segs = (p.warm > 0 || bw == 0) && n >= kMinSegmentRows && (!cyclic || n >= 2 * p.warm) ? 1 : 0;
    const int64_t extra = 2 * kMaxTileLines * sizeof(int64_t) + edge_elements(n, bw, cut) * compute_bytes;
    auto fits = [&](int64_t lpb, int64_t budget) {
        return tile_elements(n, lpb, inner) * compute_bytes + extra <= std::min<int64_t>(budget, max_lds);
    };
    // Segments for a tile of lpb lines: one per thread and line of 256
    // threads, halved while that costs few rows (fewer warm-ups), and one
    // where the warm-ups would not pay.
    auto rows = [&](int64_t segs) { return segs == 1 ? n : p.warm + ((n + segs - 1) / segs + 7) / 8 * 8; };
    auto segments = [&](int64_t lpb) -> int64_t {
        int64_t segs = kTileThreads / lpb;
        while (segs > 1 && (segs * 8 > n || rows(segs / 2) <= rows(segs) + rows(segs) / 8)) segs /= 2;
        return segs > 1 && segs >= bw && 4 * rows(segs) <= 3 * n ? segs : 1;
    };
    // Lines per tile: the least estimated time over the rounds of resident
    // workgroups.  A round copies its tiles (20 B/ns per CU; strided rows
    // move whole 64-byte sectors) and substitutes rows(segs) rows twice at
    // about 25 ns (60 cycles), workgroups on one CU sharing its SIMDs.
    // Measured against every choice from 4 to 32 lines on the grids of 1 to
    // 3 dimensions from 700 x 900 to 256^3: within 5 % of the fastest.
    double best = 0.0;
    for (int lpb = kTileLines; lpb >= 1; lpb /= 2) {
        if (!fits(lpb, 2 * kTileLdsBudget)) continue;
        if (inner >= 64 && lpb < 4) continue;  // in HBM instead
        const int64_t tiles = (p.nlines + lpb - 1) / lpb;
        const int64_t lds = tile_elements(n, lpb, inner) * compute_bytes + extra;
        const int64_t resident = std::min<int64_t>(std::min<int64_t>(3, (2 * kTileLdsBudget) / lds), (tiles + 255) / 256);
        const int64_t rounds = (tiles + 256 * resident - 1) / (256 * resident);
        const int64_t width = inner == 1 ? lpb * compute_bytes : std::max<int64_t>(lpb * compute_bytes, 64);
        const int64_t segs = cut.segs > 0 ? segments(lpb) : 1;
        const double t = rounds * resident * (2.0 * width * n / 20.0 + rows(segs) * 50.0);
        if (plan.lines == 0 || t < best) {
            best = t;
            plan.lines = lpb;
            plan.segs = cut.segs > 0 ? static_cast<int>(segs) : 0;
        }
    }
    if (plan.lines == 0) return plan;
    plan.threads = plan.segs <= 1 ? kTileThreads : std::max(64, plan.segs * plan.lines);
    return plan;
}

hipError_t launch_shift_copy(const ShiftParams& p, bool dst_f32, hipStream_t s) {
    const int64_t blocks = (p.total + kSolveBlock - 1) / kSolveBlock;
    if (blocks == 0) return hipSuccess;
    if (dst_f32)
        hipLaunchKernelGGL(shift_copy_kernel<float>, dim3(static_cast<unsigned>(blocks)), dim3(kSolveBlock), 0, s, p);
    else
        hipLaunchKernelGGL(shift_copy_kernel<double>, dim3(static_cast<unsigned>(blocks)), dim3(kSolveBlock), 0, s, p);
    return hipGetLastError();
}

}  // namespace intp_amd
