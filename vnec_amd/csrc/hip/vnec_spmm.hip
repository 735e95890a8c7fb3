// vnec_spmm.hip — several right-hand sides (k = 2, 4, 8, 16) over tiles whose
// row ends are bits (FP64 values; x [ncols][k], y [nrows][k]).
//
// A tile's nonzeros are cut into streams of R consecutive ones; a stream is
// walked by Q = min(4, k / 2) lanes, each summing k / Q right-hand sides, so a
// nonzero's x row is one contiguous piece of the load.  Each lane loads its
// share of the stream's values and columns (16 bytes at a time, laid out so
// that every load is one contiguous run of the wavefront) and the walk takes
// them from the lane that holds them by DPP: no LDS staging, no row pointers,
// no merge decisions, eight gathers in flight.  Row sums go to LDS and from
// there to y, whole rows per store, rows without nonzeros included; rows cut
// by a tile boundary are joined in the kernel as in vnec_win.hip, so the
// product is one launch.
//
// What bounds it: each x row is its own 128-byte line (k = 8 holds half of
// one).  With x rows in L2 that is the rate of the lines: the 28.7M-nonzero batch,
// k = 8, makes 30.7M requests from L1 to L2 in 185 us (165 G lines/s; bare gathers
// reach 145-177), where the merge-walking kernel this takes over from in chosen
// plans reached 135 G with its vector units half busy deciding rows.  With x
// beyond one XCD's 4 MiB of L2 it is L2's misses: uniform 4.2M, k = 4, x of 8.4 MB,
// 4.6M requests of which 2.7M miss, 347 MB in 49.6 us (7.0 TB/s).  Measured on one MI355X, replayed, that kernel at 5 items
// a thread with its carry fix-up against this one:
//   batch of 28.7M nonzeros   k = 2 187 -> 157 us, 4 199 -> 170, 8 236 -> 179
//   uniform 4.2M              k = 4 54 -> 50, 8 73.9 -> 66.7
//   R-MAT 17, 1.9M            k = 2 17.0 -> 15.6, 8 26.3 -> 20.7, 16 38 -> 28
//   banded 3.4M               k = 8 31.4 -> 19.7
//   uniform 0.09M             k = 8 12.0 -> 4.3
#include <hip/hip_runtime.h>

#include "vnec_common.h"
#include "vnec_hip.h"
#include "vnec_meet.h"
#include "vnec_offset.h"

typedef double spmm_d2 __attribute__((ext_vector_type(2)));
typedef int spmm_i4 __attribute__((ext_vector_type(4)));

template <int K> struct spmm_shape {
    static constexpr int Q = K == 2 ? 1 : K == 4 ? 2 : 4;  // lanes per stream
    static constexpr int VW = K / Q;                       // right-hand sides per lane
    static constexpr int NS = VNEC_BLOCK / Q;              // streams per tile
};

static int spmm_lanes(int k) { return k == 2 ? 1 : k == 4 ? 2 : 4; }

// ------------------------------------------------------------- builder
// Values and columns in the kernel's load order, row-end flags and first
// ordinal of each stream, row masks of the tile (see vnec_spmm_args).  The
// tile's last nonzero always carries a flag: a row left unfinished there gets
// the ordinal after the finished ones, so what the unused slots behind it add
// (0 times some x) goes nowhere.
__global__ __launch_bounds__(VNEC_BLOCK) void k_spmm_layout(
    const int32_t *__restrict__ ptr, const int32_t *__restrict__ col, const double *__restrict__ val,
    const int2 *__restrict__ co, int64_t ntiles, int Q, int R, double *__restrict__ sv, int32_t *__restrict__ sc,
    uint2 *__restrict__ sf, uint64_t *__restrict__ rmask, int32_t *__restrict__ rbase, int32_t *__restrict__ nsum)
{
    __shared__ uint32_t s_bits[VNEC_SPMM_MAX_ITEMS / 32];
    __shared__ int s_pre[VNEC_SPMM_MAX_ITEMS / 32];
    __shared__ int s_tmp[VNEC_NWAVES + 1];
    const int64_t t = blockIdx.x;
    if (t >= ntiles) return;
    const int2 c0 = co[t], c1 = co[t + 1];
    const int nrow = c1.x - c0.x, nz = c1.y - c0.y, NS = VNEC_BLOCK / Q, T = NS * R, nw = T / 32;
    const int tid = threadIdx.x;
    for (int i = tid; i < nw; i += VNEC_BLOCK) s_bits[i] = 0;
    __syncthreads();
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
            rbase[woff + (r >> 6)] = run + ex;
        }
        run += tot;
    }
    if (tid == 0) {
        const int l = nz - 1;
        if (nz > 0 && !((s_bits[l >> 5] >> (l & 31)) & 1)) {
            s_bits[l >> 5] |= 1u << (l & 31);
            run++;
        }
        nsum[t] = run;
    }
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
    for (int k = tid; k < NS; k += VNEC_BLOCK) {
        const int b = k * R, w = b >> 5, o = b & 31;
        const uint32_t f = R == 32 ? s_bits[w] : (s_bits[w] >> o) & ((1u << R) - 1u);
        sf[t * NS + k] = make_uint2(f, (uint32_t)(s_pre[w] + __popc(s_bits[w] & ((1u << o) - 1u))));
    }
    // slot d of the values: load m, stream k, lane j, element e
    for (int d = tid; d < T; d += VNEC_BLOCK) {
        const int e = d & 1, j = (d >> 1) % Q, k = (d >> 1) / Q % NS, m = (d >> 1) / (Q * NS);
        const int i = k * R + 2 * Q * m + 2 * j + e;
        sv[t * T + d] = i < nz ? val[(int64_t)c0.y + i] : 0.0;
    }
    for (int d = tid; d < T; d += VNEC_BLOCK) {
        const int e = d & 3, j = (d >> 2) % Q, k = (d >> 2) / Q % NS, m = (d >> 2) / (Q * NS);
        const int i = k * R + 4 * Q * m + 4 * j + e;
        sc[t * T + d] = i < nz ? col[(int64_t)c0.y + i] : 0;
    }
}

__global__ void k_spmm_max(const int32_t *__restrict__ a, int64_t n, int32_t *__restrict__ out)
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

extern "C" int vnec_hip_spmm_layout(const int32_t *ptr, const int32_t *col, const double *val, const int32_t *coords,
                                    int64_t ntiles, int k, int run, double *sv, int32_t *sc, uint32_t *sf,
                                    uint64_t *rmask, int32_t *rbase, int32_t *nsum, int32_t *max_dev, double *slot,
                                    void *stream)
{
    hipStream_t s = (hipStream_t)stream;
    hipLaunchKernelGGL(k_spmm_layout, dim3((unsigned)ntiles), dim3(VNEC_BLOCK), 0, s, ptr, col, val,
                       (const int2 *)coords, ntiles, spmm_lanes(k), run, sv, sc, (uint2 *)sf, rmask, rbase, nsum);
    int64_t g = (ntiles + 255) / 256;
    if (g > 256) g = 256;
    hipLaunchKernelGGL(k_spmm_max, dim3((unsigned)g), dim3(256), 0, s, (const int32_t *)nsum, ntiles, max_dev);
    hipLaunchKernelGGL(k_meet_empty, dim3((unsigned)((ntiles * k + 255) / 256)), dim3(256), 0, s, ntiles * k, 0,
                       (void *)slot);
    return (int)hipGetLastError();
}

// --------------------------------------------------------------- SpMM
// Lane j's v, in all lanes of each group of Q.
template <int Q, int J>
__device__ __forceinline__ int group_bcast(int v)
{
    if (Q == 1) return v;
    constexpr int ctrl = Q == 4 ? J * 0x55 : (J | J << 2 | (J + 2) << 4 | (J + 2) << 6);
    return __builtin_amdgcn_update_dpp(0, v, ctrl, 0xF, 0xF, true);
}
template <int Q, int J>
__device__ __forceinline__ double group_bcast(double v)
{
    if (Q == 1) return v;
    union { double d; int i[2]; } u, r;
    u.d = v;
    r.i[0] = group_bcast<Q, J>(u.i[0]);
    r.i[1] = group_bcast<Q, J>(u.i[1]);
    return r.d;
}

// Steps S .. S + U - 1 of the walk, as templates so that the source lane of
// each broadcast is a constant.
template <int K, int R, bool BIG, int S, int N>
struct spmm_gather {
    static constexpr int Q = spmm_shape<K>::Q, VW = spmm_shape<K>::VW;
    static __device__ __forceinline__ void run(const double *__restrict__ x, const spmm_i4 *C, int q,
                                               spmm_d2 (*xv)[VW / 2])
    {
        const int c = group_bcast<Q, S % (4 * Q) / 4>(C[S / (4 * Q)][S % 4]);
        const spmm_d2 *p;
        if (BIG) p = (const spmm_d2 *)(x + (int64_t)c * K + q * VW);
        else p = (const spmm_d2 *)((const char *)x + vnec_x_offset(c, K * 8, q, VW * 8));
#pragma unroll
        for (int h = 0; h < VW / 2; h++) xv[0][h] = p[h];
        spmm_gather<K, R, BIG, S + 1, N - 1>::run(x, C, q, xv + 1);
    }
};
template <int K, int R, bool BIG, int S>
struct spmm_gather<K, R, BIG, S, 0> {
    static __device__ __forceinline__ void run(const double *, const spmm_i4 *, int, spmm_d2 (*)[spmm_shape<K>::VW / 2]) {}
};

template <int K, int S, int N>
struct spmm_walk {
    static constexpr int Q = spmm_shape<K>::Q, VW = spmm_shape<K>::VW;
    static __device__ __forceinline__ void run(const spmm_d2 *V, const spmm_d2 (*xv)[VW / 2], uint32_t flags,
                                               spmm_d2 *acc, spmm_d2 *&out)
    {
        const double v = group_bcast<Q, S % (2 * Q) / 2>(V[S / (2 * Q)][S % 2]);
#pragma unroll
        for (int h = 0; h < VW / 2; h++) acc[h] += v * xv[0][h];
        if ((flags >> S) & 1) {
#pragma unroll
            for (int h = 0; h < VW / 2; h++) {
                out[h] = acc[h];
                acc[h] = 0.0;
            }
            out += K / 2;
        }
        spmm_walk<K, S + 1, N - 1>::run(V, xv + 1, flags, acc, out);
    }
};
template <int K, int S>
struct spmm_walk<K, S, 0> {
    static __device__ __forceinline__ void run(const spmm_d2 *, const spmm_d2 (*)[spmm_shape<K>::VW / 2], uint32_t,
                                               spmm_d2 *, spmm_d2 *&) {}
};

template <int K, int R, bool BIG, int S>
struct spmm_steps {
    static constexpr int VW = spmm_shape<K>::VW, U = 16 / VW;
    static __device__ __forceinline__ void run(const double *x, const spmm_i4 *C, const spmm_d2 *V, int q,
                                               uint32_t flags, spmm_d2 *acc, spmm_d2 *&out)
    {
        spmm_d2 xv[U][VW / 2];
        spmm_gather<K, R, BIG, S, U>::run(x, C, q, xv);
        spmm_walk<K, S, U>::run(V, xv, flags, acc, out);
        if constexpr (S + U < R) spmm_steps<K, R, BIG, S + U>::run(x, C, V, q, flags, acc, out);
    }
};

template <int K, int R, bool BIG>
__global__ __launch_bounds__(VNEC_BLOCK) void k_spmm_tiles(vnec_spmm_args a, int grid)
{
    constexpr int Q = spmm_shape<K>::Q, VW = spmm_shape<K>::VW, NS = spmm_shape<K>::NS, T = NS * R;
    extern __shared__ __attribute__((aligned(16))) char s_raw[];
    __shared__ uint64_t s_mask[VNEC_SPMM_MAX_ROWS / 64 + 1];
    __shared__ int s_base[VNEC_SPMM_MAX_ROWS / 64 + 1];
    __shared__ int s_f[VNEC_NWAVES];
    __shared__ double s_v[VNEC_NWAVES * K];
    spmm_d2 *s_y = (spmm_d2 *)s_raw;  // row sums, K each

    const int t = (int)xcd_tile(blockIdx.x, grid);
    if (t >= a.ntiles) return;
    const int4 d0 = ((const int4 *)a.desc)[2 * t], d1 = ((const int4 *)a.desc)[2 * t + 1];
    const int x0 = d0.x, nrow = d0.z, nz = d0.w;
    const int tid = threadIdx.x, q = tid % Q, sid = tid / Q;

    spmm_i4 C[R / (4 * Q)];
    spmm_d2 V[R / (2 * Q)];
    uint2 fo = make_uint2(0, 0);
    const bool act = sid * R < nz;
    if (act) {
        const spmm_i4 *pc = (const spmm_i4 *)(a.sc + (int64_t)t * T) + tid;
        const spmm_d2 *pv = (const spmm_d2 *)(a.sv + (int64_t)t * T) + tid;
#pragma unroll
        for (int m = 0; m < R / (4 * Q); m++) C[m] = __builtin_nontemporal_load(pc + m * VNEC_BLOCK);
#pragma unroll
        for (int m = 0; m < R / (2 * Q); m++) V[m] = __builtin_nontemporal_load(pv + m * VNEC_BLOCK);
        fo = ((const uint2 *)a.sf)[(int64_t)t * NS + sid];
    }
    const int64_t woff = (int64_t)(x0 >> 6) + t;
    if (tid * 64 < nrow) {
        s_mask[tid] = a.rmask[woff + tid];
        s_base[tid] = a.rbase[woff + tid];
    }

    spmm_d2 acc[VW / 2];
#pragma unroll
    for (int h = 0; h < VW / 2; h++) acc[h] = 0.0;
    spmm_d2 *const first = s_y + fo.y * (K / 2) + q * (VW / 2);
    if (act) {
        spmm_d2 *out = first;
        spmm_steps<K, R, BIG, 0>::run(a.x, C, V, q, fo.x, acc, out);
    }
    // rows across streams
    double tail[VW], cin[VW], incl[VW];
#pragma unroll
    for (int h = 0; h < VW; h++) tail[h] = acc[h / 2][h % 2];
    stream_seg_carry<Q, VW>(fo.x != 0, tail, s_f, s_v, cin, incl);
    if (fo.x) {
#pragma unroll
        for (int h = 0; h < VW; h++) first[h / 2][h % 2] += cin[h];
    }
    __syncthreads();
    const double *s_yd = (const double *)s_raw;
    const int64_t rstep = a.ldy ? 1 : K, cstep = a.ldy ? a.ldy : 1;  // strides of y's rows and columns
    double *y0 = a.y + x0 * rstep;
    if (tid < K) {  // rows cut by the tile's boundaries
        double *yc = y0 + tid * cstep;
        if (d1.z) meet_rows(a.slot + tid, K, d1.y, d1.z, t - d1.y, s_yd[tid], yc);
        if (d1.w)
            meet_rows(a.slot + tid, K, t, d1.w, 0, s_yd[(a.nsum[t] - 1) * K + tid], yc + nrow * rstep);
    }
    if (a.ldy) {  // column-major: a wavefront writes 64 rows of one right-hand side
        for (int c = wave_id(); c < K; c += VNEC_NWAVES)
            for (int r = (d1.z ? 1 : 0) + lane_id(); r < nrow; r += VNEC_WAVE) {
                const uint64_t m = s_mask[r >> 6];
                double o = 0.0;
                if ((m >> (r & 63)) & 1)
                    o = s_yd[(s_base[r >> 6] + __popcll(m & (((uint64_t)1 << (r & 63)) - 1))) * K + c];
                y0[c * cstep + r] = o;
            }
        return;
    }
    spmm_d2 *yr = (spmm_d2 *)y0;
    for (int i = (d1.z ? K / 2 : 0) + tid; i < nrow * (K / 2); i += VNEC_BLOCK) {
        const int r = i / (K / 2), b = r & 63;
        const uint64_t m = s_mask[r >> 6];
        spmm_d2 o = 0.0;
        if ((m >> b) & 1) {
            const int ord = s_base[r >> 6] + __popcll(m & (((uint64_t)1 << b) - 1));
            o = s_y[ord * (K / 2) + i % (K / 2)];
        }
        yr[i] = o;
    }
}

typedef void (*spmm_kernel_t)(vnec_spmm_args, int);

static spmm_kernel_t pick_spmm(int k, int run, bool big)
{
#define SK(K_, R_) \
    if (k == K_ && run == R_) return big ? k_spmm_tiles<K_, R_, true> : k_spmm_tiles<K_, R_, false>;
    SK(2, 8) SK(4, 16) SK(4, 32) SK(8, 16) SK(8, 32) SK(16, 16)
#undef SK
    return nullptr;
}

static size_t spmm_lds(const vnec_spmm_args *a) { return (size_t)a->sums * a->k * sizeof(double); }

// Row sums of a tile take 33 KiB at most (k = 8, streams of 32: 521 of them), below
// what every kernel may use without asking.
#define SPMM_LDS_MAX (40 * 1024)

extern "C" int vnec_hip_spmm_tiles(const vnec_spmm_args *a, void *stream)
{
    spmm_kernel_t k = pick_spmm(a->k, a->run, a->ncols * a->k * 8 >= ((int64_t)1 << 32));
    if (!k || spmm_lds(a) > SPMM_LDS_MAX || (((uintptr_t)a->x | (a->ldy ? 0 : (uintptr_t)a->y)) & 15)) return (int)hipErrorInvalidValue;
    if (a->ntiles <= 0) return 0;
    const int64_t grid = xcd_grid(a->ntiles);
    hipLaunchKernelGGL(k, dim3((unsigned)grid), dim3(VNEC_BLOCK), spmm_lds(a), (hipStream_t)stream, *a, (int)grid);
    return (int)hipGetLastError();
}
