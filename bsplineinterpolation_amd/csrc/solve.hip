// solve.hip -- control-point solve kernels and launchers (the device code
// is in solve_impl.hpp).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "solve_impl.hpp"

namespace intp_amd {

namespace {

template <int BW, bool CYC, typename T, typename C, int B>
__global__ __launch_bounds__(kSolveBlock) void solve_kernel(SolveParams sp) {
    const int64_t line = static_cast<int64_t>(blockIdx.x) * kSolveBlock + threadIdx.x;
    warm_factors<BW, CYC, C, kSolveBlock>(sp, sp.n);  // a few lines: all in block 0
    if (line >= sp.nlines) return;
    const int64_t o = line / sp.inner, ii = line - o * sp.inner;
    substitute<BW, CYC, C, T, B>(static_cast<T*>(sp.x) + o * sp.n * sp.inner + ii, sp.inner, sp.n, sp);
}

// Waves per SIMD the tile kernels are built for: three (168 VGPRs) where that
// does not spill, so that tiles of short lines share a CU three at a time
// (150^3 cubic, one axis: 34 us at two, 27 us at three; four spill).  Uncut
// lines have a kernel of their own, with about half the registers (orders 4
// and 7, 136^3, the contiguous axis, us: 48 and 64 as the cut kernel's plain
// path, 35 and 37); wide FP64 bands are held to three waves, or the compiler
// spends the rest on more waves and not on loads in flight (order 7, 256^3:
// 250 us unbounded, 215).
template <int BW, bool CYC, typename C, bool SEG>
constexpr int tile_waves() {
    if (!SEG) return sizeof(C) == 8 && (BW == 4 || (CYC && BW == 2)) ? 2 : 3;
    return !CYC && (sizeof(C) == 4 || BW <= 2) ? 3 : 2;
}

template <int BW, bool CYC, typename T, typename C, bool SEG>
__global__ __launch_bounds__(SEG ? kMaxTileThreads : kTileThreads)
    __attribute__((amdgpu_waves_per_eu((tile_waves<BW, CYC, C, SEG>()), !SEG && BW >= 4 && sizeof(C) == 8 ? 3 : 8))) void solve_tile_kernel(SolveParams sp) {
    extern __shared__ __align__(16) unsigned char tile_bytes[];
    __shared__ int64_t line_base[kMaxTileLines];
    const int nt = static_cast<int>(blockDim.x);  // a power of two
    solve_tile<BW, CYC, T, C, batch_rows<BW, CYC>(), SEG>(
        sp, static_cast<int64_t>(blockIdx.x) * sp.lines_per_block, tile_bytes, line_base,
        static_cast<int>(threadIdx.x + 64 * blockIdx.x) & (nt - 1), nt);
}

template <int BW, bool CYC, typename T, typename C>
hipError_t launch_lines(const SolveParams& p, int threads, hipStream_t s) {
    if (p.lines_per_block > 0) {
        const int lpb = p.lines_per_block;
        const int64_t blocks = (p.nlines + lpb - 1) / lpb;
        if (blocks > 0x7FFFFFFF) return hipErrorInvalidValue;
        const int64_t lds = tile_lds(p, BW, sizeof(C));
        if (lds + kTileStaticLds > kLdsBytes) return hipErrorInvalidValue;
        const dim3 grid(static_cast<unsigned>(blocks)), block(static_cast<unsigned>(threads));
        if (p.segs > 0)
            hipLaunchKernelGGL((solve_tile_kernel<BW, CYC, T, C, true>), grid, block, static_cast<size_t>(lds), s, p);
        else
            hipLaunchKernelGGL((solve_tile_kernel<BW, CYC, T, C, false>), grid, block, static_cast<size_t>(lds), s, p);
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
        if (lpb > kMaxTileLines || threads > (p.segs > 0 ? kMaxTileThreads : kTileThreads) || threads % lpb != 0 || threads % 64 != 0 ||
            (threads & (threads - 1)) != 0 ||
            (lpb & (lpb - 1)) != 0 || p.segs < 0 || p.segs > threads / lpb || (p.segs > 1 && p.segs < BW) || (p.segs > 0 && threads / lpb < BW) ||
            p.n >= (int64_t{1} << 24) || (p.src && p.inner != 1))
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
    int dev = 0, max_lds = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&max_lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess)
        return TilePlan{};
    return plan_tile(p, bw, cyclic, compute_bytes, max_lds);
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
