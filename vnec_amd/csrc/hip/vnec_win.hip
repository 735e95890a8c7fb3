// vnec_win.hip — windowed tiles for gfx950: merge-path SpMV whose tiles
// gather their distinct columns of x into LDS once (one right-hand side).
//
// What bounds SpMV over scattered columns here is not HBM but the 128-byte
// lines that x gathers pull from L2 into L1: a kernel that streams the nonzeros
// and gathers x once for each, no rows, moves 145-177 G lines/s with x of up to
// 4 MB, which L2 holds, 99 with x of 8 MB and 61 with 32 MB.  Lines fall with the
// number of nonzeros whose columns are sorted together, so a tile is as large as
// its x window fits LDS twice per compute unit: 512 threads x 16 nonzeros.  A
// tile holds
//   - its distinct columns, ascending (16 bits each, relative to the first of
//     every 64): gathered in that order, neighbouring lanes share lines, and
//     a column used many times in the tile is gathered once;
//   - its values and, in 16 bits, each nonzero's position in the window, in
//     CSR order, 16 to a thread, stored so that every load is one contiguous
//     run of the wavefront (values 16 bytes a lane);
//   - a bit per nonzero that ends a row, and a bit per row that has nonzeros.
// The walk is then a multiply-add and a bit test per nonzero out of registers
// and LDS: no row pointers, no search, no staged products.  Row sums go to y
// through LDS, 64 consecutive rows per store, empty rows included.  A row cut
// by a tile boundary is joined in the kernel (vnec_meet.h), so the SpMV is one
// launch.
//
// Measured on one MI355X, kernel and carry fix-up of the column-sorted plans
// used before against this kernel, us per replayed SpMV (nonzeros; FP64):
// R-MAT 18 (3.9M) 25.2 -> 17.8, power-law rows (8.0M) 63.4 -> 52.9, R-MAT 20
// (16M) 98.4 -> 78.0, 1M x 8 uniform (8.0M) 89.9 -> 63.5, 64 block-diagonal
// members (28.7M) 121.5 -> 76.8 (4.5 TB/s on the bytes it must move), 16k x 32
// uniform (0.5M) 8.4 -> 4.8, R-MAT 10 (12k) 6.8 -> 3.8.  With the gathers
// replaced by arithmetic the batch takes 62 us and R-MAT 18 11.8: what is left
// above the stream is the line traffic, partly overlapped by the other workgroup
// of the compute unit.  Requests from L1 to L2 and L2 misses by counter: R-MAT 18
// 1.8M and 0.48M in 18.0 us (101 G lines/s), the batch 8.7M and 2.8M in 80.6 (108),
// R-MAT 20 with dense rows 11.4M and 3.1M in 88.1 (130), power-law rows 7.9M and
// 1.3M in 52.6 (150).  So power-law rows and R-MAT 20 run at the rate of the bare
// gathers for their x; R-MAT 18 and the batch leave a third of it idle along a
// tile's chain of column list, gathers and walk, of which two workgroups hide each
// other's only in part.  A persistent form that loads the next
// tile during the walk (128 registers) was slower (R-MAT 18 21.7, batch 85):
// its waits cover the row stores of the tile before; tiles of 6144 items, three
// to a compute unit, lose more lines than they hide latency (R-MAT 18 20.4,
// batch 84-91); 1024 threads x 8 wait longer at each barrier (18.6, 84).
#include <hip/hip_runtime.h>

#include "vnec_common.h"
#include "vnec_hip.h"
#include "vnec_meet.h"

#define WIN_NT VNEC_WIN_THREADS
#define WIN_NW (WIN_NT / VNEC_WAVE)

// ------------------------------------------------------------- builders
// Tile boundaries: rows and nonzeros merged, eight rows weighing as much as
// row8 nonzeros, cut every `step` units, so a tile holds at most `step + snap`
// nonzeros and 8 (step + 1) / row8 + 1 rows.  W(r) = ptr[r] + r row8 / 8 is the
// weight before row r; the boundary at weight d lies in the last row with
// W <= d.  With snap > 0 a boundary fewer than snap nonzeros into a row moves
// to the row's start.
__global__ void k_win_coords(const int32_t *__restrict__ ptr, int64_t nrows, int64_t nnz, int64_t P,
                             int row8, int64_t step, int snap, int2 *__restrict__ co)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t > P) return;
    if (t == 0 || t == P) {
        co[t] = t == 0 ? make_int2(0, 0) : make_int2((int)nrows, (int)nnz);
        return;
    }
    const int64_t d = t * step;
    int64_t lo = 0, hi = nrows;  // last row with W(row) <= d
    while (lo < hi) {
        const int64_t mid = (lo + hi + 1) >> 1;
        if (ptr[mid] + mid * row8 / 8 <= d) lo = mid; else hi = mid - 1;
    }
    int64_t y = d - lo * row8 / 8;
    if (lo == nrows) {
        y = nnz;
    } else {
        if (y - ptr[lo] < snap) y = ptr[lo];
        if (y >= ptr[lo + 1]) {  // the row is complete
            y = ptr[lo + 1];
            lo++;
        }
    }
    co[t] = make_int2((int)lo, (int)y);
}

// Rows cut by tile boundaries.  meet[t] = (first tile of the row that tile t
// starts inside, that row's tiles, the tiles of the row that tile t ends
// inside, 0); a count of 0 where the boundary is a row's.
__device__ __forceinline__ int64_t win_tile_of(const int2 *co, int64_t P, int64_t j)
{
    int64_t lo = 0, hi = P - 1;  // last tile with co[tile].y <= j
    while (lo < hi) {
        const int64_t mid = (lo + hi + 1) >> 1;
        if (co[mid].y <= j) lo = mid; else hi = mid - 1;
    }
    return lo;
}

__global__ void k_win_desc(const int32_t *__restrict__ ptr, int64_t nrows, const int2 *__restrict__ co, int64_t P,
                           int4 *__restrict__ desc, const int32_t *__restrict__ nec)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= P) return;
    int4 m = make_int4(0, 0, 0, 0);
    const int2 c0 = co[t], c1 = co[t + 1];
    if (c0.x < nrows && ptr[c0.x] < c0.y) {
        const int64_t a = win_tile_of(co, P, ptr[c0.x]), b = win_tile_of(co, P, ptr[c0.x + 1] - 1);
        m.x = (int)a;
        m.y = (int)(b - a + 1);
    }
    if (c1.x < nrows && ptr[c1.x] < c1.y && (c1.x != c0.x || !m.y))
        m.z = (int)(win_tile_of(co, P, ptr[c1.x + 1] - 1) - t + 1);
    desc[2 * t] = make_int4(c0.x, c0.y, c1.x - c0.x, c1.y - c0.y);
    desc[2 * t + 1] = make_int4(nec ? nec[t] : 0, m.x, m.y, m.z);
}

// Window lists in 16 bits: per 64 entries the first column (wbase) and each
// entry's distance from it.  A tile with a distance that does not fit (a long
// row's dense piece beside a few scattered columns) is read from uniq instead:
// nec[t] gets VNEC_WIN_WIDE, and *wide is set.
__global__ __launch_bounds__(VNEC_BLOCK) void k_win_list(const int2 *__restrict__ co, int64_t ntiles,
                                                         const int32_t *__restrict__ uniq, int32_t *__restrict__ nec,
                                                         int32_t *__restrict__ wbase, uint16_t *__restrict__ woff,
                                                         int32_t *__restrict__ wide)
{
    const int64_t t = blockIdx.x;
    if (t >= ntiles) return;
    const int y0 = co[t].y, n = nec[t];
    const int64_t c0 = (int64_t)(y0 >> 6) + t;
    int bad = 0;
    for (int i = threadIdx.x; i < n; i += VNEC_BLOCK) {
        const int c = uniq[y0 + i], b = uniq[y0 + (i & ~63)];
        if ((i & 63) == 0) wbase[c0 + (i >> 6)] = b;
        woff[c0 * 64 + i] = (uint16_t)(c - b);
        bad |= c - b > 65535;
    }
    if (__syncthreads_or(bad) && threadIdx.x == 0) {
        nec[t] = n | VNEC_WIN_WIDE;
        atomicOr(wide, 1);
    }
}

// Values, window ranks, row-end flags and row masks of the tiles, in the
// order the SpMV kernel loads them; nsum[t] = LDS entries of tile t (window,
// a zero, row sums).
__global__ __launch_bounds__(VNEC_BLOCK) void k_win_layout(
    const int32_t *__restrict__ ptr, const double *__restrict__ val, const uint16_t *__restrict__ lcol,
    const int2 *__restrict__ co, int64_t ntiles, int ipt, int enc, double *__restrict__ wv,
    float *__restrict__ whi, float *__restrict__ wlo, uint16_t *__restrict__ wl, uint32_t *__restrict__ wt,
    uint64_t *__restrict__ rmask, uint16_t *__restrict__ rbase, const int32_t *__restrict__ nec,
    int32_t *__restrict__ nsum)
{
    __shared__ uint32_t s_bits[WIN_NT * VNEC_WIN_MAX_IPT / 32];
    __shared__ int s_pre[WIN_NT * VNEC_WIN_MAX_IPT / 32];
    __shared__ int s_tmp[VNEC_NWAVES + 1];
    const int64_t t = blockIdx.x;
    if (t >= ntiles) return;
    const int2 c0 = co[t], c1 = co[t + 1];
    const int nrow = c1.x - c0.x, nz = c1.y - c0.y;
    const int nt = WIN_NT, T = nt * ipt, nw = T / 32;
    const int tid = threadIdx.x;
    for (int i = tid; i < nw; i += VNEC_BLOCK) s_bits[i] = 0;
    __syncthreads();
    // rows that end in the tile with nonzeros of their own: their last
    // nonzero's flag, and per 64 rows the mask and the ordinal of the first
    const int64_t woff = (int64_t)(c0.x >> 6) + t;
    int run = 0;
    for (int base = 0; base < nrow; base += VNEC_BLOCK) {
        const int r = base + tid;
        int f = 0;
        if (r < nrow) {
            const int b = ptr[c0.x + r] - c0.y, e = ptr[c0.x + r + 1] - c0.y;
            f = e > (b > 0 ? b : 0);
            if (f) atomicOr(&s_bits[(e - 1) >> 5], 1u << ((e - 1) & 31));
        }
        const uint64_t m = __ballot(f);
        int tot;
        const int ex = block_excl_scan_i32(f, s_tmp, &tot);
        if (lane_id() == 0 && r < nrow) {
            rmask[woff + (r >> 6)] = m;
            rbase[woff + (r >> 6)] = (uint16_t)(run + ex);
        }
        run += tot;
    }
    if (tid == 0) nsum[t] = (nec[t] & ~VNEC_WIN_WIDE) + 1 + run;  // entries of LDS
    __syncthreads();
    int wrun = 0;
    for (int base = 0; base < nw; base += VNEC_BLOCK) {
        const int i = base + tid;
        int tot;
        const int ex = block_excl_scan_i32(i < nw ? __popc(s_bits[i]) : 0, s_tmp, &tot);
        if (i < nw) s_pre[i] = wrun + ex;
        wrun += tot;
    }
    __syncthreads();
    for (int k = tid; k < nt; k += VNEC_BLOCK) {
        const int b = k * ipt, w = b >> 5, o = b & 31;
        const uint32_t f = (s_bits[w] >> o) & ((1u << ipt) - 1u);
        const int ord = s_pre[w] + __popc(s_bits[w] & ((1u << o) - 1u));
        wt[t * nt + k] = f | (uint32_t)ord << 16;
    }
    // values and window ranks, thread-blocked items stored so that each load
    // of the SpMV kernel is one contiguous run of the wavefront
    const int vw = enc == 0 ? 2 : 4, lw = 4;
    const int64_t sb = t * T;
    for (int d = tid; d < T; d += VNEC_BLOCK) {
        const int q = d / vw, jj = d % vw, k = q % nt, j = (q / nt) * vw + jj;
        const int i = k * ipt + j;
        const double v = i < nz ? val[(int64_t)c0.y + i] : 0.0;
        if (enc == 0) {
            wv[sb + d] = v;
        } else {
            const float h = (float)v;
            whi[sb + d] = h;
            if (enc == 1) wlo[sb + d] = (float)(v - (double)h);
        }
    }
    for (int d = tid; d < T; d += VNEC_BLOCK) {
        const int q = d / lw, jj = d % lw, k = q % nt, j = (q / nt) * lw + jj;
        const int i = k * ipt + j;
        wl[sb + d] = i < nz ? lcol[(int64_t)c0.y + i] : (uint16_t)(nec[t] & ~VNEC_WIN_WIDE);
    }
}

__global__ void k_win_max(const int32_t *__restrict__ a, int64_t n, int32_t *__restrict__ out)
{
    int m = 0;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        m = a[i] > m ? a[i] : m;
    for (int o = 32; o > 0; o >>= 1) {
        const int v = __shfl_down(m, o, VNEC_WAVE);
        m = v > m ? v : m;
    }
    if (lane_id() == 0) atomicMax(out, m);
}

extern "C" int vnec_hip_win_coords(const int32_t *ptr, int64_t nrows, int64_t nnz, int64_t P, int row8,
                                   int64_t step, int snap, int32_t *coords, void *stream)
{
    const unsigned g = (unsigned)((P + 256) / 256);
    hipLaunchKernelGGL(k_win_coords, dim3(g), dim3(256), 0, (hipStream_t)stream, ptr, nrows, nnz, P, row8, step,
                       snap,
                       (int2 *)coords);
    return (int)hipGetLastError();
}

extern "C" int vnec_hip_win_desc(const int32_t *ptr, int64_t nrows, const int32_t *coords, int64_t ntiles,
                                 const int32_t *nec, int32_t *desc, void *stream)
{
    hipLaunchKernelGGL(k_win_desc, dim3((unsigned)((ntiles + 255) / 256)), dim3(256), 0, (hipStream_t)stream, ptr,
                       nrows, (const int2 *)coords, ntiles, (int4 *)desc, nec);
    return (int)hipGetLastError();
}

extern "C" int vnec_hip_win_list(const int32_t *coords, int64_t ntiles, const int32_t *uniq, int32_t *nec,
                                 int32_t *wbase, uint16_t *woff, int32_t *wide, void *stream)
{
    hipLaunchKernelGGL(k_win_list, dim3((unsigned)ntiles), dim3(VNEC_BLOCK), 0, (hipStream_t)stream,
                       (const int2 *)coords, ntiles, uniq, nec, wbase, woff, wide);
    return (int)hipGetLastError();
}

extern "C" int vnec_hip_win_layout(const int32_t *ptr, const double *val, const uint16_t *lcol,
                                   const int32_t *coords, int64_t ntiles, int ipt, int encoding, double *wv,
                                   float *whi, float *wlo, uint16_t *wl, uint32_t *wt, uint64_t *rmask,
                                   uint16_t *rbase, const int32_t *nec, int32_t *nsum, int32_t *max_dev, void *slot, void *stream)
{
    hipStream_t s = (hipStream_t)stream;
    const int esz = encoding == VNEC_ENC_F32_K ? 4 : 8;
    hipLaunchKernelGGL(k_win_layout, dim3((unsigned)ntiles), dim3(VNEC_BLOCK), 0, s, ptr, val, lcol,
                       (const int2 *)coords, ntiles, ipt, encoding, wv, whi, wlo, wl, wt, rmask, rbase, nec,
                       nsum);
    int64_t g = (ntiles + 255) / 256;
    if (g > 256) g = 256;
    hipLaunchKernelGGL(k_win_max, dim3((unsigned)g), dim3(256), 0, s, (const int32_t *)nsum, ntiles, max_dev);
    hipLaunchKernelGGL(k_meet_empty, dim3((unsigned)((ntiles + 255) / 256)), dim3(256), 0, s, ntiles, esz == 4, slot);
    return (int)hipGetLastError();
}

// --------------------------------------------------------------- SpMV
typedef double win_d2 __attribute__((ext_vector_type(2)));
typedef float win_f4 __attribute__((ext_vector_type(4)));
typedef uint32_t win_u4 __attribute__((ext_vector_type(4)));
typedef uint32_t win_u2 __attribute__((ext_vector_type(2)));

// A wavefront-uniform pointer kept in scalar registers, so that a load's lane
// offset needs one 32-bit register instead of a 64-bit address.
#define WIN_GLOBAL __attribute__((address_space(1)))
template <typename P>
__device__ __forceinline__ const WIN_GLOBAL P *win_uniform(const P *p)
{
    uint64_t u = (uint64_t)(uintptr_t)p;
    asm("" : "+s"(u));
    return (const WIN_GLOBAL P *)u;
}

// A thread's values of a tile as loaded.
template <int IPT, int ENC> struct WinVals;
template <int IPT> struct WinVals<IPT, 0> {
    win_d2 v[IPT / 2];
    __device__ __forceinline__ void load(const vnec_win_args &a, int64_t sb, uint32_t tid)
    {
        const win_d2 *p = (const win_d2 *)(a.wv + sb);
#pragma unroll
        for (int q = 0; q < IPT / 2; q++) v[q] = __builtin_nontemporal_load(win_uniform(p + q * WIN_NT) + tid);
    }
    __device__ __forceinline__ double get(int j) const { return v[j / 2][j % 2]; }
};
template <int IPT> struct WinVals<IPT, 1> {
    win_f4 h[IPT / 4], l[IPT / 4];
    __device__ __forceinline__ void load(const vnec_win_args &a, int64_t sb, uint32_t tid)
    {
        const win_f4 *p = (const win_f4 *)(a.whi + sb), *r = (const win_f4 *)(a.wlo + sb);
#pragma unroll
        for (int q = 0; q < IPT / 4; q++) {
            h[q] = __builtin_nontemporal_load(win_uniform(p + q * WIN_NT) + tid);
            l[q] = __builtin_nontemporal_load(win_uniform(r + q * WIN_NT) + tid);
        }
    }
    __device__ __forceinline__ double get(int j) const { return (double)h[j / 4][j % 4] + (double)l[j / 4][j % 4]; }
};
template <int IPT> struct WinVals<IPT, 2> {
    win_f4 h[IPT / 4];
    __device__ __forceinline__ void load(const vnec_win_args &a, int64_t sb, uint32_t tid)
    {
        const win_f4 *p = (const win_f4 *)(a.whi + sb);
#pragma unroll
        for (int q = 0; q < IPT / 4; q++) h[q] = __builtin_nontemporal_load(win_uniform(p + q * WIN_NT) + tid);
    }
    __device__ __forceinline__ double get(int j) const { return (double)h[j / 4][j % 4]; }
};
template <int IPT> struct WinVals<IPT, 3> {
    win_f4 h[IPT / 4];
    __device__ __forceinline__ void load(const vnec_win_args &a, int64_t sb, uint32_t tid)
    {
        const win_f4 *p = (const win_f4 *)(a.whi + sb);
#pragma unroll
        for (int q = 0; q < IPT / 4; q++) h[q] = __builtin_nontemporal_load(win_uniform(p + q * WIN_NT) + tid);
    }
    __device__ __forceinline__ float get(int j) const { return h[j / 4][j % 4]; }
};

__device__ __forceinline__ const double *win_x(const vnec_win_args &a, double) { return a.x; }
__device__ __forceinline__ const float *win_x(const vnec_win_args &a, float) { return a.x32; }
__device__ __forceinline__ double *win_y(const vnec_win_args &a, double) { return a.y; }
__device__ __forceinline__ float *win_y(const vnec_win_args &a, float) { return a.y32; }
__device__ __forceinline__ double *win_slot(const vnec_win_args &a, double) { return a.slot; }
__device__ __forceinline__ float *win_slot(const vnec_win_args &a, float) { return a.slot32; }

__device__ __forceinline__ double read_lane(double v, int l)
{
    union { double d; int i[2]; } u;
    u.d = v;
    u.i[0] = __builtin_amdgcn_readlane(u.i[0], l);
    u.i[1] = __builtin_amdgcn_readlane(u.i[1], l);
    return u.d;
}
__device__ __forceinline__ float read_lane(float v, int l)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

template <int IPT, int ENC, bool W16>
__global__ __launch_bounds__(WIN_NT) void k_spmv_win(vnec_win_args a, int grid)
{
    typedef typename enc_real<ENC>::type F;
    constexpr int T = WIN_NT * IPT, NW = WIN_NW;
    extern __shared__ __attribute__((aligned(16))) char s_raw[];
    __shared__ int s_f[NW];
    __shared__ F s_v[NW];
    const F *__restrict__ x = win_x(a, F());
    F *__restrict__ y = win_y(a, F());
    const uint32_t tid = threadIdx.x, lane = lane_id();
    const int w = __builtin_amdgcn_readfirstlane(wave_id());
    const int t = (int)xcd_tile(blockIdx.x, grid);
    if (t >= a.ntiles) return;
    const int4 d0 = ((const int4 *)a.desc)[2 * t], d1 = ((const int4 *)a.desc)[2 * t + 1];
    const int x0 = d0.x, y0 = d0.y, nrow = d0.z, nz = d0.w, nec = d1.x & ~VNEC_WIN_WIDE;
    F *s_x = (F *)s_raw;     // the x window and a zero for unused slots
    F *s_y = s_x + nec + 1;  // the tile's row sums
    F *s_pad = s_x + a.entries;

    // columns of the tile's window, in steps of four per thread; past the end
    // the last one again
    uint32_t c[IPT];
    int cbv = 0;
    const uint32_t last = nec - 1;
    if (W16 && !(d1.x & VNEC_WIN_WIDE)) {
        const int64_t ch = (int64_t)(y0 >> 6) + t;
        if (nec > 0) {
            const uint32_t q = lane * NW + w;
            cbv = win_uniform(a.wbase + ch)[q < (last >> 6) ? q : (last >> 6)];
        }
#pragma unroll
        for (int g = 0; g < IPT; g += 4)
            if (g * WIN_NT < nec) {
#pragma unroll
                for (int u = g; u < g + 4; u++) {
                    const uint32_t k = u * WIN_NT + tid;
                    c[u] = __builtin_nontemporal_load(win_uniform(a.woff + ch * 64) + (k < last ? k : last));
                }
            }
    } else {
#pragma unroll
        for (int g = 0; g < IPT; g += 4)
            if (g * WIN_NT < nec) {
#pragma unroll
                for (int u = g; u < g + 4; u++) {
                    const uint32_t k = u * WIN_NT + tid;
                    c[u] = __builtin_nontemporal_load(win_uniform(a.win + y0) + (k < last ? k : last));
                }
            }
    }
    WinVals<IPT, ENC> V;
    win_u2 lr[IPT / 4];
    uint32_t tw = 0;
    const bool act = (int)(tid * IPT) < nz;
    if (act) {
        V.load(a, (int64_t)t * T, tid);
        const win_u2 *p = (const win_u2 *)(a.wl + (int64_t)t * T);
#pragma unroll
        for (int q = 0; q < IPT / 4; q++) lr[q] = __builtin_nontemporal_load(win_uniform(p + q * WIN_NT) + tid);
        tw = __builtin_nontemporal_load(win_uniform(a.wt + (int64_t)t * WIN_NT) + tid);
    }
    // row masks of the tile, 64 words of 64 rows per wavefront
    const int64_t woff = (int64_t)(x0 >> 6) + t;
    uint64_t ml = 0;
    int bl = 0;
    if ((int)(w + NW * lane) * VNEC_WAVE < nrow) {
        ml = a.rmask[woff + w + NW * lane];
        bl = a.rbase[woff + w + NW * lane];
    }
    // the gathers, all in flight: one wait for the columns (vmcnt(0)), since
    // the compiler, which cannot count loads issued under the conditions
    // above, would otherwise wait before each gather for the one before it
    F xv[IPT];
    __builtin_amdgcn_s_waitcnt(0x0F70);
#pragma unroll
    for (int g = 0; g < IPT; g += 4)
        if (g * WIN_NT < nec) {
#pragma unroll
            for (int u = g; u < g + 4; u++) {
                if (W16) {  // (x below 4 GiB: 32-bit byte offsets)
                    const WIN_GLOBAL char *xb =
                        (const WIN_GLOBAL char *)win_uniform(x + __builtin_amdgcn_readlane(cbv, u));
                    xv[u] = *(const WIN_GLOBAL F *)(xb + c[u] * (uint32_t)sizeof(F));
                } else {
                    xv[u] = x[c[u]];
                }
            }
        }
    __builtin_amdgcn_s_waitcnt(0x0F70);
#pragma unroll
    for (int g = 0; g < IPT; g += 4)
        if (g * WIN_NT < nec) {
#pragma unroll
            for (int u = g; u < g + 4; u++) *((int)(u * WIN_NT + tid) < nec ? s_x + u * WIN_NT + tid : s_pad) = xv[u];
        }
    if (tid == 0) s_x[nec] = 0;
    __syncthreads();

    // walk: rows that end among the thread's items
    int flags = 0, ord0 = 0;
    F acc = 0;
    if (act) {
        flags = tw & 0xFFFF;
        ord0 = tw >> 16;
        int ord = ord0;
#pragma unroll
        for (int q = 0; q < IPT / 4; q++) {
            F xs[4];
#pragma unroll
            for (int e = 0; e < 4; e++) xs[e] = s_x[(lr[q][e / 2] >> (16 * (e % 2))) & 0xFFFF];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int j = 4 * q + e;
                acc += V.get(j) * xs[e];
                if ((flags >> j) & 1) {
                    s_y[ord++] = acc;
                    acc = 0;
                }
            }
        }
    }
    // partial rows join across threads
    int f = flags != 0;
    F v = acc;
    wave_seg_scan(f, v);
    if (lane == VNEC_WAVE - 1) {
        s_f[w] = f;
        s_v[w] = v;
    }
    __syncthreads();
    F cw = 0;  // carry into this wavefront
    {
        int wf = 0;
        F wv = 0;
        if (lane < NW) {
            wf = s_f[lane];
            wv = s_v[lane];
        }
        wave_seg_scan(wf, wv);
        if (w > 0) cw = read_lane(wv, w - 1);
    }
    const F blk = f ? v : v + cw;
    const F cin = wave_shift_up1(blk, cw);
    if (flags) s_y[ord0] += cin;
    F *slot = win_slot(a, F());
    if (tid == WIN_NT - 1) {  // the tile's last, partial row
        if (d1.w) meet_rows(slot, 1, t, d1.w, 0, blk, y + x0 + nrow);
        else if (d1.z && nrow == 0) meet_rows(slot, 1, d1.y, d1.z, t - d1.y, blk, y + x0);
    }
    __syncthreads();
    if (tid == 0 && d1.z && nrow > 0)  // its first row, begun in an earlier tile
        meet_rows(slot, 1, d1.y, d1.z, t - d1.y, s_y[0], y + x0);

    // the tile's rows, 64 at a time
    for (int q0 = w; q0 * VNEC_WAVE < nrow; q0 += NW * VNEC_WAVE) {
        if (q0 != w) {
            const int ql = q0 + NW * lane;
            if (ql * VNEC_WAVE < nrow) {
                ml = a.rmask[woff + ql];
                bl = a.rbase[woff + ql];
            }
        }
        for (int k = 0; k < VNEC_WAVE; k++) {
            const int q = q0 + NW * k;
            if (q * VNEC_WAVE >= nrow) break;
            const uint32_t mlo = __builtin_amdgcn_readlane((int)(uint32_t)ml, k);
            const uint32_t mhi = __builtin_amdgcn_readlane((int)(uint32_t)(ml >> 32), k);
            const int base = __builtin_amdgcn_readlane(bl, k);
            const int r = q * VNEC_WAVE + lane;
            const int o = __builtin_amdgcn_mbcnt_hi(mhi, __builtin_amdgcn_mbcnt_lo(mlo, 0u));
            const uint32_t half = lane < 32 ? mlo : mhi;
            F out = 0;
            if ((half >> (lane & 31)) & 1) out = s_y[base + o];
            if (r < nrow && !(r == 0 && d1.z)) y[x0 + r] = out;
        }
    }
}

typedef void (*win_kernel_t)(vnec_win_args, int);

static win_kernel_t pick_win(int ipt, int enc, bool w16)
{
#define WE(I, E) \
    if (ipt == I && enc == E) return w16 ? k_spmv_win<I, E, true> : k_spmv_win<I, E, false>;
#define WC(I) WE(I, 0) WE(I, 1) WE(I, 2) WE(I, 3)
    WC(4) WC(8) WC(16)
    return nullptr;
#undef WC
#undef WE
}

static size_t win_lds(const vnec_win_args *a)
{
    return (size_t)(a->entries + 1) * (a->encoding == VNEC_ENC_F32_K ? sizeof(float) : sizeof(double));
}

// The most a tile of this kernel can need: its nonzeros all in columns of
// their own and each a row's last.
static size_t win_lds_max(const vnec_win_args *a)
{
    return (size_t)(2 * WIN_NT * a->ipt + 2) * (a->encoding == VNEC_ENC_F32_K ? sizeof(float) : sizeof(double));
}

// The limit is the kernel's, not the plan's: the same value whichever plan
// asks, so that no plan lowers it under another one's launches.
extern "C" int vnec_hip_win_prepare(const vnec_win_args *a)
{
    win_kernel_t k = pick_win(a->ipt, a->encoding, a->woff != nullptr);
    if (!k) return (int)hipErrorInvalidValue;
    return (int)hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)win_lds_max(a));
}

extern "C" int vnec_hip_spmv_win(const vnec_win_args *a, void *stream)
{
    win_kernel_t k = pick_win(a->ipt, a->encoding, a->woff != nullptr);
    if (!k || win_lds(a) > win_lds_max(a)) return (int)hipErrorInvalidValue;
    if (a->ntiles <= 0) return 0;
    const int64_t grid = xcd_grid(a->ntiles);
    hipLaunchKernelGGL(k, dim3((unsigned)grid), dim3(WIN_NT), win_lds(a), (hipStream_t)stream, *a, (int)grid);
    return (int)hipGetLastError();
}
