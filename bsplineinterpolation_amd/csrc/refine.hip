// refine.hip -- FP64 residuals for the refined-FP32 build.
//
// The control points c (FP32) of a refined build solve
//     (M_0 (x) M_1 (x) ... (x) M_{D-1}) c = S f
// where M_d is dimension d's collocation matrix (the unfactored matrix the
// reference factors, InterpolationTemplate.hpp:254-446) and S f the values
// with the periodic index shift (InterpolationTemplate.hpp:452-462).  A
// refinement sweep forms r = S f - (M_0 (x) ... ) c in FP64 (band mat-vecs
// along the axes: the FP64 counterpart of the reference's BandMatrix
// product, BandMatrix.hpp:68-77, 148-172; all axes in one pass where that is
// faster, otherwise one axis at a time), solves for the correction in FP32
// with the LU factors, and adds it to c.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "kernels.hpp"

namespace intp_amd {

namespace {

constexpr int kBlock = 256;

// One output element per thread.  The table is viewed as (outer, n, inner)
// along the applied axis; indices use 32-bit arithmetic (tables below
// 2^32 elements) and multiply-high divisions by the invariant extents.
// The half-width W is a template argument so that the 2W+1 loads of a
// row are all issued before the first product.
// With xcd_remap, each XCD takes a contiguous range of blocks, so that
// the blocks of neighbouring rows (which share 2W of their 2W+1 input
// rows) meet in one L2; otherwise block b goes to XCD b mod 8.
template <int W, typename TI, typename TO>
__global__ __launch_bounds__(kBlock) void band_matvec_kernel(MatvecParams p) {
    const uint64_t blk = p.xcd_remap ? static_cast<uint64_t>(xcd_chunk_index()) : blockIdx.x;
    const uint64_t e64 = blk * kBlock + threadIdx.x;
    if (e64 >= static_cast<uint64_t>(p.total)) return;
    const uint32_t e = static_cast<uint32_t>(e64);
    const uint32_t n = static_cast<uint32_t>(p.n), inner = static_cast<uint32_t>(p.inner);
    const uint32_t t = fast_div(e, p.div_inner);
    const uint32_t j = t - fast_div(t, p.div_n) * n;
    const uint32_t base = e - j * inner;
    const TI* __restrict__ x = static_cast<const TI*>(p.x);
    const double* __restrict__ row = p.colloc + j * static_cast<uint32_t>(2 * W + 1);
    // out-of-range columns of a clamped dimension read element j and count
    // as zero (their matrix entries are zero too)
    double xv[2 * W + 1];
#pragma unroll
    for (int m = -W; m <= W; ++m) {
        int64_t jj = static_cast<int64_t>(j) + m;
        bool ok = true;
        if (p.periodic) {
            jj = jj < 0 ? jj + n : jj >= n ? jj - n : jj;
        } else {
            ok = jj >= 0 && jj < n;
            jj = ok ? jj : j;
        }
        const double v = static_cast<double>(x[base + static_cast<uint32_t>(jj) * inner]);
        xv[m + W] = ok ? v : 0.0;
    }
    double acc = 0.0;
#pragma unroll
    for (int m = 0; m <= 2 * W; ++m) acc += row[m] * xv[m];
    if (p.src) {
        // residual: the shifted value minus the product; element
        // (i_0..i_{D-1}) reads source element ((i_d - shift_d) mod n_d)
        uint32_t rem = e;
        uint64_t src = 0, mul = 1;
        for (int d = p.dim - 1; d >= 0; --d) {
            const uint32_t nd = static_cast<uint32_t>(p.dn[d]);
            const uint32_t qd = fast_div(rem, p.div_dn[d]);
            const uint32_t id = rem - qd * nd;
            rem = qd;
            int64_t s = static_cast<int64_t>(id) - p.dshift[d];
            if (s < 0) s += nd;
            src += static_cast<uint64_t>(s) * mul;
            mul *= nd;
        }
        acc = p.src[src] - acc;
    }
    static_cast<TO*>(p.y)[e] = static_cast<TO>(acc);
}

// Row-run variant for the axes before the last (inner > 1): a thread
// takes R consecutive rows j0..j0+R-1 of one column (o, i) and slides a
// window of R + 2W loaded values along them, so an input element is
// loaded (R + 2W) / R times instead of 2W + 1.  Consecutive threads take
// consecutive i (coalesced).  Each output sums its products in the order
// of band_matvec_kernel, so the results are the same.
// Requires n > 2W: a periodic index then needs at most one wrap.
template <int W, int R, typename TI, typename TO>
__global__ __launch_bounds__(kBlock) void band_matvec_rows_kernel(MatvecParams p) {
    const uint64_t blk = p.xcd_remap ? static_cast<uint64_t>(xcd_chunk_index()) : blockIdx.x;
    const uint64_t w64 = blk * kBlock + threadIdx.x;
    if (w64 >= static_cast<uint64_t>(p.work)) return;
    const uint32_t w = static_cast<uint32_t>(w64);
    const uint32_t n = static_cast<uint32_t>(p.n), inner = static_cast<uint32_t>(p.inner);
    const uint32_t t = fast_div(w, p.div_inner);
    const uint32_t i = w - t * inner;
    const uint32_t o = fast_div(t, p.div_runs);
    const uint32_t j0 = (t - o * static_cast<uint32_t>(p.runs)) * R;
    const uint32_t rows = min(static_cast<uint32_t>(R), n - j0);
    const uint32_t base = o * n * inner + i;
    const TI* __restrict__ x = static_cast<const TI*>(p.x);
    // window entry q holds element j0 - W + q; entries past the last row's
    // stencil, and out-of-range columns of a clamped dimension (whose
    // matrix entries are zero), read element j0 and count as zero
    double xv[R + 2 * W];
#pragma unroll
    for (int q = 0; q < R + 2 * W; ++q) {
        int64_t jj = static_cast<int64_t>(j0) - W + q;
        bool ok = static_cast<uint32_t>(q) < rows + 2 * W;
        if (p.periodic) {
            jj = jj < 0 ? jj + n : jj >= n ? jj - n : jj;
        } else {
            ok = ok && jj >= 0 && jj < n;
        }
        jj = ok ? jj : j0;
        const double v = static_cast<double>(x[base + static_cast<uint32_t>(jj) * inner]);
        xv[q] = ok ? v : 0.0;
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        if (static_cast<uint32_t>(r) >= rows) break;
        const uint32_t j = j0 + r;
        const uint32_t e = base + j * inner;
        const double* __restrict__ row = p.colloc + j * static_cast<uint32_t>(2 * W + 1);
        double acc = 0.0;
#pragma unroll
        for (int m = 0; m <= 2 * W; ++m) acc += row[m] * xv[r + m];
        if (p.src) {
            uint32_t rem = e;
            uint64_t src = 0, mul = 1;
            for (int d = p.dim - 1; d >= 0; --d) {
                const uint32_t nd = static_cast<uint32_t>(p.dn[d]);
                const uint32_t qd = fast_div(rem, p.div_dn[d]);
                const uint32_t id = rem - qd * nd;
                rem = qd;
                int64_t s = static_cast<int64_t>(id) - p.dshift[d];
                if (s < 0) s += nd;
                src += static_cast<uint64_t>(s) * mul;
                mul *= nd;
            }
            acc = p.src[src] - acc;
        }
        static_cast<TO*>(p.y)[e] = static_cast<TO>(acc);
    }
}

// The residual of a 2D or 3D table in one pass.  A workgroup owns a tile of
// kResRows x 64 positions of dimensions 1 and 2 and walks a chunk of
// dimension 0 plane by plane: the plane's tile of c, with its halo, goes to
// LDS; the products along dimension 2 (a thread's column is fixed, its matrix
// row stays in registers) go to LDS again; those along dimension 1 run down a
// thread's kResR rows (the matrix rows are the same for a wave: scalar
// loads); and along dimension 0 every plane adds its term to the 2W + 1
// results still open, held in registers.  The sums take the products in the
// order of the kernels above, so the results are the same bits.
// Plane p is loaded, p - 1 multiplied along dimension 2 and p - 2 along 1 and
// 0 between two barriers, each from its own half of the buffers.
// Against three passes over FP64 tables (0.67 GB at 256^3) this one moves
// c, the values and the result, 0.27 GB.  256^3, order 5: 281 -> 113 us, of
// which the FP64 products at full rate take 35 and the traffic 55; one
// workgroup a CU (156 VGPRs) leaves the barriers and LDS waits between.
constexpr int kResWaves = 8;
constexpr int kResR = 4;
constexpr int kResRows = kResWaves * kResR;
constexpr int kResThreads = kResWaves * 64;

template <int K, int D>
__global__ __launch_bounds__(kResThreads) void residual_kernel(ResidualParams p) {
    constexpr int W = K > 1 ? K - 1 : 0, WP = K / 2;  // clamped, periodic half-widths
    constexpr int ROWS = kResRows + 2 * W, COLS = 64 + 2 * W, TILE = ROWS * COLS;
    constexpr int PER = (TILE + kResThreads - 1) / kResThreads;
    constexpr int WROWS = (ROWS + kResWaves - 1) / kResWaves;
    typedef const __attribute__((address_space(4))) double* Uniform;
    __shared__ float xs[2][TILE];
    __shared__ double ys[2][ROWS * 64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n0 = p.n[0], n1 = p.n[1], n2 = p.n[2];
    uint32_t b = static_cast<uint32_t>(xcd_chunk_index());
    const int t2 = static_cast<int>(b % static_cast<uint32_t>(p.tiles2));
    b /= static_cast<uint32_t>(p.tiles2);
    const int t1 = static_cast<int>(b % static_cast<uint32_t>(p.tiles1));
    const int j0 = static_cast<int>(b / static_cast<uint32_t>(p.tiles1)) * p.chunk;
    const int j1 = min(n0, j0 + p.chunk);
    const int first1 = t1 * kResRows, first2 = t2 * 64;
    const int row0 = first1 + wave * kResR, col = first2 + lane;

    // wrapped index of a periodic dimension, or -1 outside
    auto element = [](int i, int n, int periodic) {
        if (periodic) i = i < 0 ? i + n : i >= n ? i - n : i;
        return i >= 0 && i < n ? i : -1;
    };
    // the thread's elements of a plane's tile
    int64_t off[PER];
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        const int e = threadIdx.x + q * kResThreads;
        const int r = element(first1 - W + e / COLS, n1, p.periodic[1]);
        const int c = element(first2 - W + e % COLS, n2, p.periodic[2]);
        off[q] = e < TILE && r >= 0 && c >= 0 ? static_cast<int64_t>(r) * n2 + c : -1;
    }
    // the matrix row of the thread's column, in the middle of 2W + 1 entries
    double m2[2 * W + 1];
#pragma unroll
    for (int m = -W; m <= W; ++m) {
        const int w = p.w[2];
        const int64_t at = static_cast<int64_t>(min(col, n2 - 1)) * (2 * w + 1) + m + w;
        m2[m + W] = m >= -w && m <= w ? p.colloc[2][at] : 0.0;
    }
    // sources of the thread's results, less their plane
    int64_t from[kResR];
#pragma unroll
    for (int r = 0; r < kResR; ++r) {
        int s1 = row0 + r - p.shift[1], s2 = col - p.shift[2];
        s1 += s1 < 0 ? n1 : 0;
        s2 += s2 < 0 ? n2 : 0;
        from[r] = static_cast<int64_t>(s1) * n2 + s2;
    }
    const int64_t plane = static_cast<int64_t>(n1) * n2;
    const int w0 = p.w[0], w1 = p.w[1], w2 = p.w[2];
    const int begin = j0 - w0, end = j1 + w0;  // planes (outside [0, n0): wrapped, or zeros)

    float next[PER];
    auto load = [&](int pl) {
        const int g = pl < end ? element(pl, n0, p.periodic[0]) : -1;
        const float* __restrict__ x = p.c + static_cast<int64_t>(max(g, 0)) * plane;
#pragma unroll
        for (int q = 0; q < PER; ++q) next[q] = g >= 0 && off[q] >= 0 ? x[off[q]] : 0.f;
    };
    auto store = [&](int pl) {
        float* x = xs[pl & 1];
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            const int e = threadIdx.x + q * kResThreads;
            if (e < TILE) x[e] = next[q];
        }
    };
    // along dimension 2, half-width w of W
    auto along2 = [&](int pl, auto width) {
        constexpr int w = decltype(width)::value;
        const float* x = xs[pl & 1] + lane + (W - w);
        double* y = ys[pl & 1] + lane;
#pragma unroll
        for (int q = 0; q < WROWS; ++q) {
            const int r = q * kResWaves + wave;
            if (r >= ROWS) break;
            double acc = 0.0;
#pragma unroll
            for (int m = 0; m <= 2 * w; ++m) acc += m2[W - w + m] * static_cast<double>(x[r * COLS + m]);
            y[r * 64] = acc;
        }
    };
    double y1[kResR];
    auto along1 = [&](int pl, auto width) {
        constexpr int w = decltype(width)::value;
        const double* y = ys[pl & 1] + (wave * kResR + W - w) * 64 + lane;
        double v[kResR + 2 * w];
#pragma unroll
        for (int q = 0; q < kResR + 2 * w; ++q) v[q] = y[q * 64];
#pragma unroll
        for (int r = 0; r < kResR; ++r) {
            const Uniform row = (Uniform)p.colloc[1] + static_cast<int64_t>(min(row0 + r, n1 - 1)) * (2 * w + 1);
            double acc = 0.0;
#pragma unroll
            for (int m = 0; m <= 2 * w; ++m) acc += row[m] * v[r + m];
            y1[r] = acc;
        }
    };
    // open results along dimension 0: sum[i] belongs to plane pl - w + i
    double sum[D == 3 ? 2 * W + 1 : 1][kResR];
#pragma unroll
    for (auto& s : sum)
#pragma unroll
        for (int r = 0; r < kResR; ++r) s[r] = 0.0;
    auto along0 = [&](int pl, auto width) {
        constexpr int w = decltype(width)::value;
#pragma unroll
        for (int i = 0; i <= 2 * w; ++i) {
            const int j = min(max(pl - w + i, 0), n0 - 1);
            const double m = ((Uniform)p.colloc[0])[static_cast<int64_t>(j) * (2 * w + 1) + 2 * w - i];
#pragma unroll
            for (int r = 0; r < kResR; ++r) sum[i][r] += m * y1[r];
        }
    };
    auto emit = [&](int j, const double (&src)[kResR], const double (&v)[kResR]) {
#pragma unroll
        for (int r = 0; r < kResR; ++r)
            if (row0 + r < n1 && col < n2)
                p.out[j * plane + static_cast<int64_t>(row0 + r) * n2 + col] = static_cast<float>(src[r] - v[r]);
    };

    load(begin);
    store(begin);
    load(begin + 1);
    __syncthreads();
    for (int pl = begin; pl <= end; ++pl) {
        // plane pl + 1 to LDS, pl along dimension 2, pl - 1 along 1 and 0
        store(pl + 1);
        load(pl + 2);
        const int done = pl - 1 - w0;  // the result that plane pl - 1 completes
        double src[kResR];
        if (done >= j0) {
            int s0 = done - p.shift[0];
            s0 += s0 < 0 ? n0 : 0;
#pragma unroll
            for (int r = 0; r < kResR; ++r)
                src[r] = row0 + r < n1 && col < n2 ? p.src[s0 * plane + from[r]] : 0.0;
        }
        if (pl < end) {
            if (w2 == W)
                along2(pl, std::integral_constant<int, W>{});
            else
                along2(pl, std::integral_constant<int, WP>{});
        }
        if (pl > begin) {
            if (w1 == W)
                along1(pl - 1, std::integral_constant<int, W>{});
            else
                along1(pl - 1, std::integral_constant<int, WP>{});
            if constexpr (D == 3) {
                if (w0 == W)
                    along0(pl - 1, std::integral_constant<int, W>{});
                else
                    along0(pl - 1, std::integral_constant<int, WP>{});
                if (done >= j0) emit(done, src, sum[0]);
#pragma unroll
                for (int i = 0; i < 2 * W; ++i)
#pragma unroll
                    for (int r = 0; r < kResR; ++r) sum[i][r] = sum[i + 1][r];
#pragma unroll
                for (int r = 0; r < kResR; ++r) sum[w0 == W ? 2 * W : 2 * WP][r] = 0.0;
            } else {
                emit(0, src, y1);
            }
        }
        __syncthreads();
    }
}

__global__ __launch_bounds__(kBlock) void add_f32_kernel(float* __restrict__ c, const float* __restrict__ d,
                                                         int64_t total) {
    const int64_t e = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
    if (e < total) c[e] = c[e] + d[e];
}

// Gradient-table cells of element e: c = c0 + delta in FP64 (exact: the
// correction is far below c0's last bit), the backward differences of
// those sums along each dimension, each rounded once to FP32; and c itself.
// Neighbouring blocks share their rows and planes, so each XCD takes a
// contiguous range of blocks, and the cells are streamed past L2.  256^3 (0.47
// GB moved): 147 us, and 35 for c in a pass of its own -> 108 us; 156 us
// without the streaming stores.
template <int D, typename C>
__global__ __launch_bounds__(kBlock) void refined_cells_kernel(CellParams p) {
    const uint64_t e64 = static_cast<uint64_t>(xcd_chunk_index()) * kBlock + threadIdx.x;
    if (e64 >= static_cast<uint64_t>(p.total)) return;
    const uint32_t e = static_cast<uint32_t>(e64);
    const float* __restrict__ c0 = p.c0;
    const float* __restrict__ delta = p.delta;
    auto full = [&](uint32_t i) {
        double v = static_cast<double>(c0[i]);
        if (delta) v += static_cast<double>(delta[i]);
        return v;
    };
    const double c = full(e);
    float diff[3] = {0.f, 0.f, 0.f};
    uint32_t rem = e, stride = 1;
#pragma unroll
    for (int d = D - 1; d >= 0; --d) {
        const uint32_t nd = static_cast<uint32_t>(p.n[d]);
        const uint32_t q = fast_div(rem, p.div_n[d]);
        const uint32_t id = rem - q * nd;
        rem = q;
        if (id > 0)
            diff[d] = static_cast<float>(c - full(e - stride));
        else if (p.periodic[d])
            diff[d] = static_cast<float>(c - full(e + (nd - 1) * stride));
        stride *= nd;
    }
    C out;
    out.c = static_cast<float>(c);
    out.e0 = diff[0];
    if constexpr (D >= 2) {
        out.e1 = diff[1];
        out.e2 = diff[2];
    }
    if constexpr (D >= 2) {
        // streamed past the rows and planes that the next blocks read again
        typedef float f32x4 __attribute__((ext_vector_type(4)));
        static_assert(sizeof(C) == sizeof(f32x4), "a cell is one 16-byte store");
        __builtin_nontemporal_store(f32x4{out.c, out.e0, out.e1, out.e2}, static_cast<f32x4*>(p.cells) + e);
    } else {
        static_cast<C*>(p.cells)[e] = out;
    }
    if (p.c) p.c[e] = out.c;
}

constexpr int kRunRows = 8;

template <int W>
hipError_t launch_matvec_width(const MatvecParams& p, bool in_f32, bool out_f32, int64_t blocks, hipStream_t s) {
    const dim3 block(kBlock);
    if (p.runs > 0) {
        const dim3 grid(static_cast<unsigned>((p.work + kBlock - 1) / kBlock));
        if (in_f32 && out_f32)
            hipLaunchKernelGGL((band_matvec_rows_kernel<W, kRunRows, float, float>), grid, block, 0, s, p);
        else if (in_f32)
            hipLaunchKernelGGL((band_matvec_rows_kernel<W, kRunRows, float, double>), grid, block, 0, s, p);
        else if (out_f32)
            hipLaunchKernelGGL((band_matvec_rows_kernel<W, kRunRows, double, float>), grid, block, 0, s, p);
        else
            hipLaunchKernelGGL((band_matvec_rows_kernel<W, kRunRows, double, double>), grid, block, 0, s, p);
        return hipGetLastError();
    }
    const dim3 grid(static_cast<unsigned>(blocks));
    if (in_f32 && out_f32)
        hipLaunchKernelGGL((band_matvec_kernel<W, float, float>), grid, block, 0, s, p);
    else if (in_f32)
        hipLaunchKernelGGL((band_matvec_kernel<W, float, double>), grid, block, 0, s, p);
    else if (out_f32)
        hipLaunchKernelGGL((band_matvec_kernel<W, double, float>), grid, block, 0, s, p);
    else
        hipLaunchKernelGGL((band_matvec_kernel<W, double, double>), grid, block, 0, s, p);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_band_matvec(const MatvecParams& p_in, bool in_f32, bool out_f32, hipStream_t s) {
    if (p_in.total >= (int64_t{1} << 32)) return hipErrorInvalidValue;
    MatvecParams p = p_in;
    p.div_inner = make_fast_div(static_cast<uint32_t>(p.inner));
    p.div_n = make_fast_div(static_cast<uint32_t>(p.n));
    for (int d = 0; d < p.dim && d < kMaxDim; ++d) p.div_dn[d] = make_fast_div(static_cast<uint32_t>(p.dn[d]));
    // the blocks of rows j and j+1 are inner / kBlock apart: under the
    // default round-robin over 8 XCDs they share an L2 only when that
    // distance is a multiple of 8
    p.xcd_remap = p.inner > 1 && (p.inner % kBlock != 0 || (p.inner / kBlock) % 8 != 0) ? 1 : 0;
    const int64_t blocks = (p.total + kBlock - 1) / kBlock;
    if (blocks == 0) return hipSuccess;
    // axes before the last take the row-run kernel
    p.runs = 0;
    p.work = 0;
    if (p.inner > 1 && p.n > 2 * static_cast<int64_t>(p.w)) {
        p.runs = static_cast<int32_t>((p.n + kRunRows - 1) / kRunRows);
        p.div_runs = make_fast_div(static_cast<uint32_t>(p.runs));
        p.work = p.total / p.n * p.runs;
    }
    switch (p.w) {
        case 0: return launch_matvec_width<0>(p, in_f32, out_f32, blocks, s);
        case 1: return launch_matvec_width<1>(p, in_f32, out_f32, blocks, s);
        case 2: return launch_matvec_width<2>(p, in_f32, out_f32, blocks, s);
        case 3: return launch_matvec_width<3>(p, in_f32, out_f32, blocks, s);
        case 4: return launch_matvec_width<4>(p, in_f32, out_f32, blocks, s);
        case 5: return launch_matvec_width<5>(p, in_f32, out_f32, blocks, s);
        case 6: return launch_matvec_width<6>(p, in_f32, out_f32, blocks, s);
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_residual(int dim, int order, const ResidualParams& p_in, hipStream_t s) {
    ResidualParams p = p_in;
    if (dim < 2 || dim > 3 || order < 1 || order > 7 || (dim == 2 && p.n[0] != 1)) return hipErrorInvalidValue;
    const int w = order > 1 ? order - 1 : 0;
    for (int d = 3 - dim; d < 3; ++d)
        if (p.n[d] < 1 || p.w[d] != (p.periodic[d] ? order / 2 : w) || (p.periodic[d] && p.n[d] < 2 * p.w[d] + 1))
            return hipErrorInvalidValue;
    p.tiles1 = (p.n[1] + kResRows - 1) / kResRows;
    p.tiles2 = (p.n[2] + 63) / 64;
    // chunks along dimension 0: as many workgroups as the 256 CUs hold (two
    // each up to order 4, by registers), down to three planes a chunk: each
    // multiplies 2 w planes again, but a small table leaves CUs idle (builds,
    // at least 8 planes -> 3: 32^3, order 5, 108 -> 97 us; 100^3, order 5, 172
    // -> 159 us; cubic 145 -> 136 us)
    const int64_t tiles = static_cast<int64_t>(p.tiles1) * p.tiles2;
    const int64_t fill = (order <= 4 ? 512 : 256) / tiles;
    const int64_t chunks = std::max<int64_t>(1, std::min<int64_t>(fill, p.n[0] / 3));
    p.chunk = static_cast<int32_t>((p.n[0] + chunks - 1) / chunks);
    const int64_t blocks = tiles * ((p.n[0] + p.chunk - 1) / p.chunk);
    if (blocks > 0x7FFFFFFF) return hipErrorInvalidValue;
    const dim3 grid(static_cast<unsigned>(blocks)), block(kResThreads);
#define RESIDUAL_CASE(K)                                                          \
    case K:                                                                       \
        if (dim == 2)                                                             \
            hipLaunchKernelGGL((residual_kernel<K, 2>), grid, block, 0, s, p);    \
        else                                                                      \
            hipLaunchKernelGGL((residual_kernel<K, 3>), grid, block, 0, s, p);    \
        return hipGetLastError();
    switch (order) {
        RESIDUAL_CASE(1)
        RESIDUAL_CASE(2)
        RESIDUAL_CASE(3)
        RESIDUAL_CASE(4)
        RESIDUAL_CASE(5)
        RESIDUAL_CASE(6)
        RESIDUAL_CASE(7)
        default: return hipErrorInvalidValue;
    }
#undef RESIDUAL_CASE
}

hipError_t launch_refined_cells(const CellParams& p_in, hipStream_t s) {
    if (p_in.total >= (int64_t{1} << 32) || p_in.dim < 1 || p_in.dim > kCellMaxDim || p_in.c == p_in.c0) return hipErrorInvalidValue;
    CellParams p = p_in;
    int64_t total = 1;
    for (int d = 0; d < p.dim; ++d) {
        p.div_n[d] = make_fast_div(static_cast<uint32_t>(p.n[d]));
        total *= p.n[d];
    }
    if (total != p.total) return hipErrorInvalidValue;
    const int64_t blocks = (p.total + kBlock - 1) / kBlock;
    if (blocks == 0) return hipSuccess;
    const dim3 grid(static_cast<unsigned>(blocks)), block(kBlock);
    switch (p.dim) {
        case 1: hipLaunchKernelGGL((refined_cells_kernel<1, Cell1>), grid, block, 0, s, p); break;
        case 2: hipLaunchKernelGGL((refined_cells_kernel<2, Cell3>), grid, block, 0, s, p); break;
        default: hipLaunchKernelGGL((refined_cells_kernel<3, Cell3>), grid, block, 0, s, p); break;
    }
    return hipGetLastError();
}

hipError_t launch_add_f32(float* c, const float* d, int64_t total, hipStream_t s) {
    const int64_t blocks = (total + kBlock - 1) / kBlock;
    if (blocks == 0) return hipSuccess;
    hipLaunchKernelGGL(add_f32_kernel, dim3(static_cast<unsigned>(blocks)), dim3(kBlock), 0, s, c, d, total);
    return hipGetLastError();
}

}  // namespace intp_amd
