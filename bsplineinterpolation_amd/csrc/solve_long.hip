// solve_long.hip -- control-point solve of lines too long for LDS (a 1D
// spline of 20,000 points and more, a strided axis of a few thousand): the
// line is cut into chunks of rows, one workgroup each, and a chunk into
// segments, one lane each, with the warm-up and the comparisons of
// solve_segments (solve_impl.hpp) at both kinds of cuts.
//
//   1. forward: every chunk substitutes its rows into `tmp`, from the state
//      its own warm-up arrives at, and records that state and its last rows;
//   2. join forward: one thread per line compares each chunk's starting
//      state with its neighbour's last rows, bit for bit, and substitutes a
//      chunk again, row by row, where they differ; for cyclic lines it then
//      sums the strips and solves the last rows, which fix the corners;
//   3. backward: every chunk, from `tmp` into the table;
//   4. join backward: as 2, in the other direction.
// Each sweep reads one array and writes another, so a chunk can be solved
// again from unchanged rows.  The results are those of the sequential
// substitution, bit for bit.
//
// One lane used to walk such a line in HBM: every row waited for its chain
// (about 100 cycles) and its share of the factor loads.  1D cubic, n =
// 100,000, kernels of the solve: 10,050 -> 28 us (forward 11.6, backward
// 11.1, the joins 2.8 each), bound by the warm-ups of 56 rows and the
// launches.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "solve_impl.hpp"

namespace intp_amd {

namespace {

template <typename C>
struct LongParams {
    SolveParams sp;
    C* tmp;        // the table's shape: forward results
    C* state;      // [4][chunks][nlines][BW]: forward start, end; backward start, end
    C* vmax;       // [chunks][nlines]: largest forward |row| (cyclic)
    C* corner;     // [nlines][BW] (cyclic)
    int32_t chunks, rows, len, segs;
};

template <typename C>
__device__ __forceinline__ C* state_at(const LongParams<C>& p, int kind, int chunk, int64_t line, int bw) {
    return p.state + ((static_cast<int64_t>(kind) * p.chunks + chunk) * p.sp.nlines + line) * bw;
}

// Element offset of row 0 of a line in the table, and in the first pass's
// values (shifted dims, as in solve_tile).
__device__ __forceinline__ int64_t table_base(const SolveParams& sp, int64_t line) {
    const int64_t o = line / sp.inner;
    return o * sp.n * sp.inner + (line - o * sp.inner);
}

__device__ __forceinline__ int64_t values_base(const SolveParams& sp, int64_t line) {
    int64_t rem = line, off = 0, mul = sp.n;
#pragma unroll
    for (int d = kMaxDim - 1; d >= 0; --d) {
        if (d >= sp.outer_dims) continue;
        const int64_t nd = sp.outer_n[d];
        const int64_t id = rem % nd;
        rem /= nd;
        int64_t w = id - sp.outer_shift[d];
        if (w < 0) w += nd;
        off += w * mul;
        mul *= nd;
    }
    return off;
}

// Right-hand side of row j of a line.
template <typename T, typename C>
__device__ __forceinline__ C source_row(const SolveParams& sp, int64_t base, int64_t j) {
    if (sp.src) {
        int64_t js = j - sp.shift_last;
        if (js < 0) js += sp.n;
        return static_cast<C>(sp.src[base + js]);
    }
    return static_cast<C>(static_cast<const T*>(sp.x)[base + j * sp.inner]);
}

// The chunk's workgroup: rows [origin, origin + rows) of lines first ..
// first + nl - 1 into the tile, row-major with `step` elements a row.
template <typename F, typename C>
__device__ __forceinline__ void fill_tile(C* tile, int step, int lpb, int nl, int64_t origin, int rows, int64_t end,
                                          int NT, F row_of) {
    constexpr int U = 8;
    const int shift = __builtin_ctz(static_cast<unsigned>(lpb));
    const int l = static_cast<int>(threadIdx.x) & (lpb - 1);
    const int per = NT >> shift;
    for (int r0 = static_cast<int>(threadIdx.x) >> shift; r0 < rows; r0 += per * U) {
        C v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t j = origin + r0 + u * per;
            v[u] = l < nl && r0 + u * per < rows && j >= 0 && j < end ? row_of(l, j) : C(0);
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (r0 + u * per < rows) tile[(r0 + u * per) * step + l] = v[u];
    }
}

template <int BW, bool CYC, typename T, typename C>
__global__ __launch_bounds__(256) void long_forward_kernel(LongParams<C> p) {
    constexpr int B = batch_rows<BW, CYC>();
    extern __shared__ __align__(16) unsigned char bytes[];
    __shared__ int64_t base[kMaxTileLines];
    __shared__ int64_t src_base[kMaxTileLines];
    __shared__ int failed;
    const SolveParams& sp = p.sp;
    const int NT = static_cast<int>(blockDim.x), tid = static_cast<int>(threadIdx.x);
    const int lpb = sp.lines_per_block, step = static_cast<int>(tile_step(lpb, sp.inner));
    const int64_t first = static_cast<int64_t>(blockIdx.y) * lpb;
    const int nl = static_cast<int>(min(static_cast<int64_t>(lpb), sp.nlines - first));
    const int chunk = static_cast<int>(blockIdx.x), r0 = chunk * p.rows, warm = sp.warm;
    const int n = static_cast<int>(sp.n), H = CYC ? n - BW : n;
    if (tid < nl) {
        base[tid] = table_base(sp, first + tid);
        src_base[tid] = sp.src ? values_base(sp, first + tid) : base[tid];
    }
    __syncthreads();
    // rows r0 - warm .. r0 + rows - 1 and a pad on both sides
    const int pad = static_cast<int>(kTilePad), origin = r0 - warm;
    C* tile = reinterpret_cast<C*>(bytes) + pad * step;
    const int held = p.rows + warm + 2 * pad, limit = min(H, r0 + p.rows);
    auto load = [&]() {
        fill_tile(tile - pad * step, step, lpb, nl, static_cast<int64_t>(origin) - pad, held, static_cast<int64_t>(H), NT,
                  [&](int l, int64_t j) { return source_row<T, C>(sp, src_base[l], j); });
        __syncthreads();
    };
    const EdgeTable<C> edge = stage_edges<BW, C>(sp, reinterpret_cast<C*>(bytes) + held * step, tid, NT);
    load();
    const int shift = __builtin_ctz(static_cast<unsigned>(lpb));
    const int line = tid & (lpb - 1), seg = tid >> shift;
    C* x = tile + line;
    C start[BW + 1], hist[BW + 1], vmax = C(0);
    for (int attempt = 0;; ++attempt) {
        const int segs = attempt == 0 ? p.segs : 1, len = attempt == 0 ? p.len : p.rows;
        const int a = r0 + seg * len;
        const bool mine = line < nl && seg < segs && a < H;
        const int wave = __builtin_amdgcn_readfirstlane(tid) & ~63;
        const int seg0 = wave >> shift, seg1 = min((wave + 63) >> shift, min(segs, (H - r0 + len - 1) / len) - 1);
#pragma unroll
        for (int m = 0; m <= BW; ++m) hist[m] = C(0);
        vmax = C(0);
        if (tid == 0) failed = 0;
        seg_forward<BW, CYC, false, C, B>(x, step, origin, limit, a - warm, warm, H, mine && a > 0,
                                          equal_batches(seg0, seg1, len, warm - r0, warm, sp.flo, sp.fhi, H, B), sp,
                                          edge, hist, vmax);
#pragma unroll
        for (int m = 0; m < BW; ++m) start[m] = hist[m];
        __syncthreads();
        seg_forward<BW, CYC, true, C, B>(x, step, origin, limit, a, len, H, mine,
                                         equal_batches(seg0, seg1, len, -r0, len, sp.flo, sp.fhi, H, B), sp, edge,
                                         hist, vmax);
        __syncthreads();
        bool bad = false;
        if (mine && seg > 0) {
#pragma unroll
            for (int m = 0; m < BW; ++m) bad = bad || !same_bits(start[m], x[(a - 1 - m - origin) * step]);
        }
        if (__any(bad) && (tid & 63) == 0) failed = 1;
        __syncthreads();
        const bool again = failed != 0;
        if (!again) break;  // one segment has no cuts: the second attempt ends here
        load();
    }
    // results, the chunk's states and its largest row
    const int end = min(r0 + p.rows, H);
    {
        const int per = NT >> shift;
        if (line < nl)
            for (int j = r0 + (tid >> shift); j < end; j += per)
                p.tmp[base[line] + static_cast<int64_t>(j) * sp.inner] = x[(j - origin) * step];
    }
    if (line < nl && seg == 0) {
        C* st = state_at(p, 0, chunk, first + line, BW);
        C* en = state_at(p, 1, chunk, first + line, BW);
#pragma unroll
        for (int m = 0; m < BW; ++m) {
            st[m] = start[m];
            en[m] = x[(end - 1 - m - origin) * step];
        }
    }
    if constexpr (CYC && BW > 0) {
        // largest |row| per line; non-negative FP64 numbers order like their
        // bits, infinities and NaN (which a row keeps to its segment's end)
        // above all
        __shared__ unsigned long long big[kMaxTileLines];
        if (tid < lpb) big[tid] = 0;
        __syncthreads();
        const double v = hist[0] - hist[0] == C(0) ? static_cast<double>(vmax) : fabs(static_cast<double>(hist[0]));
        if (line < nl && (tid >> shift) * p.len + r0 < H)
            atomicMax(&big[line], static_cast<unsigned long long>(__double_as_longlong(v)));
        __syncthreads();
        if (tid < nl)
            p.vmax[static_cast<int64_t>(chunk) * sp.nlines + first + tid] =
                static_cast<C>(__longlong_as_double(static_cast<long long>(big[tid])));
    }
}

// Whether every chunk of a line starts from its neighbour's last rows (a
// wave per line, a lane per cut).
template <int BW, typename C>
__device__ __forceinline__ bool cuts_agree(const LongParams<C>& p, int kind, int64_t line) {
    bool same = true;
    for (int c = 1 + static_cast<int>(threadIdx.x); c < p.chunks; c += 64) {
        const C* st = state_at(p, kind, c, line, BW);
        const C* before = state_at(p, kind + 1, c - 1, line, BW);
#pragma unroll
        for (int m = 0; m < BW; ++m) same = same && same_bits(st[m], before[m]);
    }
    return __all(same);
}

template <int BW, typename C>
__device__ __forceinline__ bool cut_agrees(const LongParams<C>& p, int kind, int c, int64_t line) {
    const C* st = state_at(p, kind, c, line, BW);
    const C* before = state_at(p, kind + 1, c - 1, line, BW);
    bool same = true;
#pragma unroll
    for (int m = 0; m < BW; ++m) same = same && same_bits(st[m], before[m]);
    return same;
}

// One wave per line.
template <int BW, bool CYC, typename T, typename C>
__global__ __launch_bounds__(64) void long_join_forward_kernel(LongParams<C> p) {
#pragma clang fp contract(off)
    constexpr int B = batch_rows<BW, CYC>();
    const SolveParams& sp = p.sp;
    const int64_t line = blockIdx.x;
    const int lane = static_cast<int>(threadIdx.x);
    const int64_t n = sp.n, H = CYC ? n - BW : n;
    const int64_t base = table_base(sp, line), src_base = sp.src ? values_base(sp, line) : base;
    const int32_t z = lane_zero();
    LineState<BW, CYC, C> st;
#pragma unroll
    for (int m = 0; m <= BW; ++m) st.hist[m] = st.nxt[m] = st.corner[m] = st.acc[m] = C(0);
    if (!cuts_agree<BW>(p, 0, line)) {
        for (int c = 1; c < p.chunks; ++c) {
            if (cut_agrees<BW>(p, 0, c, line)) continue;
            const int64_t r0 = static_cast<int64_t>(c) * p.rows, end = min(r0 + p.rows, H);
            for (int64_t j = r0 + lane; j < end; j += 64)
                p.tmp[base + j * sp.inner] = source_row<T, C>(sp, src_base, j);
            __threadfence_block();
            __syncthreads();
            if (lane == 0) {
                const C* before = state_at(p, 1, c - 1, line, BW);
                LineState<BW, false, C> sf;  // the strips follow below
#pragma unroll
                for (int m = 0; m <= BW; ++m) sf.hist[m] = sf.nxt[m] = sf.corner[m] = sf.acc[m] = C(0);
#pragma unroll
                for (int m = 0; m < BW; ++m) sf.hist[m] = before[m];
                forward_range<BW, false, C, C, B>(p.tmp + base, sp.inner, n, r0, end, sp, sf, z);
                C* en = state_at(p, 1, c, line, BW);
#pragma unroll
                for (int m = 0; m < BW; ++m) en[m] = sf.hist[m];
            }
            __threadfence_block();
            __syncthreads();
            if constexpr (CYC) {
                C big = C(0);
                for (int64_t j = r0 + lane; j < end; j += 64) {
                    const C v = fabs(p.tmp[base + j * sp.inner]);
                    big = v > big || v != v ? v : big;
                    if (big != big) break;
                }
#pragma unroll
                for (int o = 32; o > 0; o >>= 1) {
                    const C v = __shfl_xor(big, o, 64);
                    big = v > big || v != v ? v : big;
                }
                if (lane == 0) p.vmax[static_cast<int64_t>(c) * sp.nlines + line] = big;
                __threadfence_block();
                __syncthreads();
            }
        }
    }
    if constexpr (CYC && BW > 0) {
        C big = C(0);
        for (int c = lane; c < p.chunks; c += 64) {
            const C v = p.vmax[static_cast<int64_t>(c) * sp.nlines + line];
            big = v > big || v != v ? v : big;
            if (big != big) break;
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            const C v = __shfl_xor(big, o, 64);
            big = v > big || v != v ? v : big;
        }
        // the strips' leading terms, then lane q sums strip q
        __shared__ C term[BW * 256];
        const C* __restrict__ bottom = static_cast<const C*>(sp.bottom);
        const int prefix = min(sp.warm, 256);
        for (int i = lane; i < BW * prefix; i += 64) {
            const int q = i / prefix, j = i - q * prefix;
            term[i] = bottom[static_cast<int64_t>(q) * n + j] * p.tmp[base + static_cast<int64_t>(j) * sp.inner];
        }
        __shared__ C sum[BW];
        __syncthreads();
        if (lane < BW) {
            const int q = lane;
            const int64_t last = n - 2 * BW + q;
            C a = source_row<T, C>(sp, src_base, H + q);
            int64_t j = 0;
#pragma unroll 8
            for (; j < prefix; ++j) a = a - term[q * prefix + j];
            const C t = static_cast<C>(sp.strip_rest) * big;
            if (!(big - big == C(0)) || !(a - t == a && a + t == a) || same_bits(a, C(-0.0)) || prefix < sp.warm)
                for (; j < last; ++j) a = a - bottom[q * n + j] * p.tmp[base + j * sp.inner];
            sum[q] = a;
        }
        __syncthreads();
        if (lane != 0) return;
        // the last rows, then the backward rows that fix the corners
#pragma unroll
        for (int m = 0; m < BW; ++m) {
            st.hist[m] = p.tmp[base + (H - 1 - m) * sp.inner];
            st.acc[m] = sum[m];
            p.tmp[base + (H + m) * sp.inner] = C(0);
        }
        forward_range<BW, CYC, C, C, 1>(p.tmp + base, sp.inner, n, H, n, sp, st, z);
        backward_range<BW, CYC, C, C, 1>(p.tmp + base, sp.inner, n, H, n, sp, st, z);
#pragma unroll
        for (int m = 0; m < BW; ++m) p.corner[line * BW + m] = st.corner[m];
    }
}

template <int BW, bool CYC, typename T, typename C>
__global__ __launch_bounds__(256) void long_backward_kernel(LongParams<C> p) {
    constexpr int B = batch_rows<BW, CYC>();
    extern __shared__ __align__(16) unsigned char bytes[];
    __shared__ int64_t base[kMaxTileLines];
    __shared__ int failed;
    const SolveParams& sp = p.sp;
    const int NT = static_cast<int>(blockDim.x), tid = static_cast<int>(threadIdx.x);
    const int lpb = sp.lines_per_block, step = static_cast<int>(tile_step(lpb, sp.inner));
    const int64_t first = static_cast<int64_t>(blockIdx.y) * lpb;
    const int nl = static_cast<int>(min(static_cast<int64_t>(lpb), sp.nlines - first));
    const int n = static_cast<int>(sp.n), H = CYC ? n - BW : n, warm = sp.warm;
    // chunks from the end: rows [e0 - rows, e0)
    const int chunk = static_cast<int>(blockIdx.x), e0 = H - chunk * p.rows;
    if (tid < nl) base[tid] = table_base(sp, first + tid);
    __syncthreads();
    const int pad = static_cast<int>(kTilePad), origin = e0 - p.rows;
    C* tile = reinterpret_cast<C*>(bytes) + pad * step;
    const int held = p.rows + warm + 2 * pad;
    auto load = [&]() {
        fill_tile(tile - pad * step, step, lpb, nl, static_cast<int64_t>(origin) - pad, held, static_cast<int64_t>(H),
                  NT, [&](int l, int64_t j) { return p.tmp[base[l] + j * sp.inner]; });
        __syncthreads();
    };
    const EdgeTable<C> edge = stage_edges<BW, C>(sp, reinterpret_cast<C*>(bytes) + held * step, tid, NT);
    load();
    const int shift = __builtin_ctz(static_cast<unsigned>(lpb));
    const int line = tid & (lpb - 1), seg = tid >> shift;
    C* x = tile + line;
    C corner[BW + 1];
    corner[BW] = C(0);
#pragma unroll
    for (int c = 0; c < BW; ++c) corner[c] = CYC && line < nl ? p.corner[(first + line) * BW + c] : C(0);
    const KnownDivisor<C> kz = known_pivot<C>(sp);
    const int blo = H - min(sp.bhi, H), bhi = H - sp.blo;
    C start[BW + 1], nxt[BW + 1];
    nxt[BW] = C(0);
    for (int attempt = 0;; ++attempt) {
        const int segs = attempt == 0 ? p.segs : 1, len = attempt == 0 ? p.len : p.rows;
        const int top = e0 - seg * len;
        const bool mine = line < nl && seg < segs && top > 0;
        const int wave = __builtin_amdgcn_readfirstlane(tid) & ~63;
        const int seg0 = wave >> shift, seg1 = min((wave + 63) >> shift, min(segs, (e0 + len - 1) / len) - 1);
        const int before = H - e0;
#pragma unroll
        for (int m = 0; m < BW; ++m) nxt[m] = CYC && top + warm >= H ? corner[m] : C(0);
        if (tid == 0) failed = 0;
        seg_backward<BW, CYC, false, C, B>(x, step, origin, n, top + warm - 1, warm, H, mine && top < H,
                                           equal_batches(seg0, seg1, len, warm - before, warm, blo, bhi, H, B), sp,
                                           edge, kz, corner, nxt);
#pragma unroll
        for (int m = 0; m < BW; ++m) start[m] = nxt[m];
        __syncthreads();
        seg_backward<BW, CYC, true, C, B>(x, step, origin, n, top - 1, len, H, mine,
                                          equal_batches(seg0, seg1, len, -before, len, blo, bhi, H, B), sp, edge, kz,
                                          corner, nxt);
        __syncthreads();
        bool bad = false;
        if (mine && seg > 0) {
#pragma unroll
            for (int m = 0; m < BW; ++m) bad = bad || !same_bits(start[m], x[(top + m - origin) * step]);
        }
        if (__any(bad) && (tid & 63) == 0) failed = 1;
        __syncthreads();
        const bool again = failed != 0;
        if (!again) break;  // one segment has no cuts: the second attempt ends here
        load();
    }
    T* __restrict__ X = static_cast<T*>(sp.x);
    const int from = max(origin, 0);
    {
        const int per = NT >> shift;
        if (line < nl)
            for (int j = from + (tid >> shift); j < e0; j += per)
                X[base[line] + static_cast<int64_t>(j) * sp.inner] = static_cast<T>(x[(j - origin) * step]);
    }
    if (line < nl && seg == 0) {
        C* st = state_at(p, 2, chunk, first + line, BW);
        C* en = state_at(p, 3, chunk, first + line, BW);
#pragma unroll
        for (int m = 0; m < BW; ++m) {
            st[m] = start[m];
            en[m] = x[(from + m - origin) * step];
        }
        if (CYC && chunk == 0) {
#pragma unroll
            for (int m = 0; m < BW; ++m) X[base[line] + static_cast<int64_t>(H + m) * sp.inner] = static_cast<T>(corner[m]);
        }
    }
}

// One wave per line; a chunk is solved again in place in tmp, whose rows no
// other chunk reads any more.
template <int BW, bool CYC, typename T, typename C>
__global__ __launch_bounds__(64) void long_join_backward_kernel(LongParams<C> p) {
    constexpr int B = batch_rows<BW, CYC>();
    const SolveParams& sp = p.sp;
    const int64_t line = blockIdx.x;
    const int lane = static_cast<int>(threadIdx.x);
    if (cuts_agree<BW>(p, 2, line)) return;
    const int64_t n = sp.n, H = CYC ? n - BW : n;
    const int64_t base = table_base(sp, line);
    T* __restrict__ X = static_cast<T*>(sp.x);
    const int32_t z = lane_zero();
    LineState<BW, CYC, C> st;
#pragma unroll
    for (int m = 0; m <= BW; ++m) st.hist[m] = st.nxt[m] = st.corner[m] = st.acc[m] = C(0);
    if constexpr (CYC) {
#pragma unroll
        for (int m = 0; m < BW; ++m) st.corner[m] = p.corner[line * BW + m];
    }
    for (int c = 1; c < p.chunks; ++c) {
        if (cut_agrees<BW>(p, 2, c, line)) continue;
        const int64_t e0 = H - static_cast<int64_t>(c) * p.rows, from = max(e0 - p.rows, int64_t{0});
        if (lane == 0) {
            const C* before = state_at(p, 3, c - 1, line, BW);
#pragma unroll
            for (int m = 0; m < BW; ++m) st.nxt[m] = before[m];
            backward_range<BW, CYC, C, C, B>(p.tmp + base, sp.inner, n, from, e0, sp, st, z);
            C* en = state_at(p, 3, c, line, BW);
#pragma unroll
            for (int m = 0; m < BW; ++m) en[m] = st.nxt[m];
        }
        __threadfence_block();
        __syncthreads();
        for (int64_t j = from + lane; j < e0; j += 64) X[base + j * sp.inner] = static_cast<T>(p.tmp[base + j * sp.inner]);
        __syncthreads();
    }
}

template <typename C>
size_t long_state_bytes(const SolveParams& p, int bw, const LongShape& s) {
    const size_t lines = static_cast<size_t>(p.nlines);
    return (lines * (static_cast<size_t>(s.chunks) * (4 * bw + 1) + bw) + 1) * sizeof(C);
}

template <int BW, bool CYC, typename T, typename C>
hipError_t launch_long(const SolveParams& sp, void* scratch, hipStream_t s) {
    const LongShape shape = plan_long(sp, BW, CYC, sizeof(C));
    if (shape.lpb == 0) return hipErrorInvalidValue;
    LongParams<C> p{};
    p.sp = sp;
    p.sp.lines_per_block = shape.lpb;
    p.sp.segs = shape.segs;
    p.chunks = shape.chunks;
    p.rows = shape.rows;
    p.len = shape.len;
    p.segs = shape.segs;
    const size_t lines = static_cast<size_t>(sp.nlines);
    p.tmp = static_cast<C*>(scratch);
    p.state = p.tmp + lines * static_cast<size_t>(sp.n);
    p.vmax = p.state + 4 * lines * shape.chunks * BW;
    p.corner = p.vmax + lines * shape.chunks;
    const int64_t groups = (sp.nlines + shape.lpb - 1) / shape.lpb;
    if (groups > 65535 || sp.nlines > 0x7FFFFFFF || sp.n >= (int64_t{1} << 28)) return hipErrorInvalidValue;
    const size_t lds = static_cast<size_t>(long_lds(p.sp, BW, shape, sizeof(C)));
    const dim3 grid(static_cast<unsigned>(shape.chunks), static_cast<unsigned>(groups)), block(shape.threads);
    const dim3 lgrid(static_cast<unsigned>(sp.nlines));
    hipLaunchKernelGGL((long_forward_kernel<BW, CYC, T, C>), grid, block, lds, s, p);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;  // the others read what it writes
    if (BW > 0) hipLaunchKernelGGL((long_join_forward_kernel<BW, CYC, T, C>), lgrid, dim3(64), 0, s, p);
    hipLaunchKernelGGL((long_backward_kernel<BW, CYC, T, C>), grid, block, lds, s, p);
    if (BW > 0) hipLaunchKernelGGL((long_join_backward_kernel<BW, CYC, T, C>), lgrid, dim3(64), 0, s, p);
    return hipGetLastError();
}

template <int BW, typename T, typename C>
hipError_t launch_long_bw(bool cyclic, const SolveParams& p, void* scratch, hipStream_t s) {
    if (!cyclic) return launch_long<BW, false, T, C>(p, scratch, s);
    if constexpr (2 * BW <= kMaxOrder) return launch_long<BW, true, T, C>(p, scratch, s);
    return hipErrorNotSupported;
}

template <typename T, typename C>
hipError_t launch_long_typed(int bw, bool cyclic, const SolveParams& p, void* scratch, hipStream_t s) {
    switch (bw) {
        case 0: return launch_long_bw<0, T, C>(cyclic, p, scratch, s);
        case 1: return launch_long_bw<1, T, C>(cyclic, p, scratch, s);
        case 2: return launch_long_bw<2, T, C>(cyclic, p, scratch, s);
        case 3: return launch_long_bw<3, T, C>(cyclic, p, scratch, s);
        case 4: return launch_long_bw<4, T, C>(cyclic, p, scratch, s);
        case 5: return launch_long_bw<5, T, C>(cyclic, p, scratch, s);
        case 6: return launch_long_bw<6, T, C>(cyclic, p, scratch, s);
        default: return hipErrorNotSupported;
    }
}

}  // namespace

// Bounds the scratch of a long-line solve (its forward results are a second
// table); larger ones are solved in place, one lane per line.
constexpr int64_t kLongScratchMax = int64_t{1} << 30;

size_t solve_long_scratch(const SolveParams& p, int bw, bool cyclic, int compute_bytes) {
    if ((p.warm == 0 && bw > 0) || p.n >= (int64_t{1} << 28) || (cyclic && p.n < 2 * p.warm)) return 0;
    const LongShape s = plan_long(p, bw, cyclic, compute_bytes);
    // a chunk at least, and every warm-up inside the line it warms up on
    if (s.lpb == 0 || s.chunks < 2 || (p.nlines + s.lpb - 1) / s.lpb > 65535) return 0;
    if (p.nlines > kLongScratchMax / compute_bytes / p.n) return 0;
    const size_t state = compute_bytes == 4 ? long_state_bytes<float>(p, bw, s) : long_state_bytes<double>(p, bw, s);
    return static_cast<size_t>(p.nlines) * static_cast<size_t>(p.n) * compute_bytes + state;
}

hipError_t launch_solve_long(int bw, bool cyclic, SolveTypes types, const SolveParams& p, void* scratch,
                             hipStream_t s) {
    if (p.accum) return hipErrorInvalidValue;
    switch (types) {
        case SolveTypes::kF64: return launch_long_typed<double, double>(bw, cyclic, p, scratch, s);
        case SolveTypes::kF32: return launch_long_typed<float, float>(bw, cyclic, p, scratch, s);
        case SolveTypes::kF32StoreF64Compute: return launch_long_typed<float, double>(bw, cyclic, p, scratch, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace intp_amd
