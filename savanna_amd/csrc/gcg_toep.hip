// Matrix-core kernels for the shapes the tile family of gcg_mfma.hip does not take: groups of any width (down to one
// channel per filter), filters of 9 to 256 taps, tensors of any element alignment.
//
// There is one filter per channel at worst, so the columns of a product cannot be channels that share a filter.
// They are blocks of time instead: with t = 16 n + m a channel's convolution is the matrix product
//     y2[m, n] = sum_k A[m, k] U[k, n],   A[m, k] = h~[m - k + OFF],   U[k, n] = u[16 n + k - OFF]
// (h~ by lag, OFF = 32 NK - 16), 16 x 16 outputs of one channel from NK 32-deep products.  A lane's operand of U is 8
// consecutive samples at a multiple of 8, one aligned 16-byte LDS read once u lies channel-major; the Toeplitz
// operand is 8 consecutive taps at any offset, read as five words and shifted by half a word where the offset is odd.
// The anti-causal product of the backward is the same with U[k, n] = g2[16 n + k], A[m, k] = h~[k - m].  The filter
// gradient is one more product per channel, all lags in one tile: with lag = 16 a + b
//     dh~[a, b] = sum_s G[a, s] V[s, b],   G[a, s] = g2[s + 16 a],   V[s, b] = u[s - b]
// so the accumulator of a channel is four registers whatever the filter length (up to 256).
//
// Precision is that of the fp32 vector kernels of gcg_direct.hip: every operand enters as a sum of bf16 planes that
// hold it exactly (the product of two bf16 values has 16 significant bits: two planes; of two f16 values 22: three;
// fp32: three), and of the plane products those with m + n <= 2 are formed; the ones left out are below 2^-24.
// A matrix instruction rounds its sum towards minus infinity, not to the nearest value: in a product of 32 NK terms
// that is below the vector kernels' own error, but in the filter gradient, a sum over all rows, it adds up to a bias
// (dh 2.5 to 6 times as far from 64 bits as the vector kernels'; 1 x 16384 x (16 groups of 32), 256 taps: 1.8e-6 of the
// 2-norm against 3.2e-7).  There each instruction's chain is 32 rows long, a tile and a run are summed on the vector
// ALUs, and half of a tile's products enter negated, so that the bias of one half is taken off by the other's: 1.4e-7,
// and below the vector kernels' error at every shape compared, for 4 % of the backward's time.
//
// Infinities, NaN, samples and taps from 2^104 on, results from 2^80 on (LIFT): the products multiply samples with the zeros
// around the band, and a plane of such a value is infinite or NaN.  Whatever the sample, some y2 or du of the run is then not finite;
// a workgroup that met one does its run once more on the vector ALUs, tap by tap in fp32 and with the sums of the filter
// gradient cut the same way: a sample then reaches the rows its taps reach and no other.  Looking at the results costs
// 1 % of the kernels' time, at the samples (their largest magnitude) 4 %.
//
// A workgroup owns CB adjacent channels and a run of 256-row tiles of one batch row; u (and g2) of a tile and of the
// filter's reach stay in LDS as rings, so each row is read once (dy twice in the backward: for g2 OFF rows ahead, and
// for dC).  Measured at 1 x 4096 x (256 groups of 8), 128 taps, bf16, against gcg_direct.hip: forward 124 -> 22 us,
// backward 333 -> 63 us, its filter-gradient sum 27 -> 4 us.  What bounds it (SQ counters there): vector instructions --
// the split into planes, its transposition between the tensors' channel-fastest rows and the channel-major rings, one
// access per element -- take 44 % of the SIMDs' issue cycles forward and 56 % backward, matrix instructions occupy 13 and
// 22 %, and waves spend half of their time waiting, for rows and at the two or four barriers of a tile.  Memory is far off:
// 71 MB in 22 us forward, 146 MB in 63 us backward.
#include "gcg_mfma_tile.h"

#include <type_traits>

namespace gcg {
namespace {

constexpr int TT = 256;                          // time rows per tile: 16 blocks of 16
constexpr int YP = TT + 4;                       // floats per channel of the result tile (16-byte accesses of 16 channels hit 64 banks)

template <typename T> struct GT;                 // planes of an activation and of a filter operand
template <> struct GT<float> { static constexpr int NPA = 3, NPW = 3; };
template <> struct GT<bf16_t> { static constexpr int NPA = 2, NPW = 1; };
template <> struct GT<f16_t> { static constexpr int NPA = 3, NPW = 2; };
template <> struct GT<bf16w_t> { static constexpr int NPA = 2, NPW = 3; };
template <> struct GT<f16w_t> { static constexpr int NPA = 3, NPW = 3; };

// Samples enter the rings and taps the tables times 2^24, and results are divided by both: the last planes of a value below
// 2^-110 would be bf16 subnormals, and bits of it lost (f16's smallest tap is 2^-24 and its smallest product 2^-48: no need)
template <typename T> constexpr float LIFT = std::is_same_v<T, f16_t> || std::is_same_v<T, f16w_t> ? 1.f : 0x1p24f;
template <typename T> constexpr float DROP = 1.f / (LIFT<T> * LIFT<typename Filt<T>::type>);       // of y2 and du

template <int NK> struct Reach {
    static constexpr int OFF = 32 * NK - 16;     // rows of history (u) and look-ahead (g2) held beside a tile
    static constexpr int R = TT + OFF;           // ring length
    static constexpr int RP = R + 8;             // pitch: the first 8 samples are repeated behind the last
    static constexpr int HP = 32 * NK + 24;      // pitch of a tap table
};

// LDS bytes of a workgroup of cb channels touching nf filters; dirs = 1 (forward) or 2 (backward: two rings, two tables)
constexpr int lds_bytes(int npa, int npw, int nk, int cb, int nf, int dirs)
{
    return 16 + dirs * npa * cb * (TT + 32 * nk - 16 + 8) * 2 + cb * YP * 4 + dirs * npw * nf * (32 * nk + 24) * 2;
}
constexpr int LDS_MAX = 160 * 1024;
// 32 channels (64-byte rows at 16 bits, 16 waves) where the rings and one filter per channel fit, else 16
constexpr int pick_cb(int npa, int npw, int nk, int dirs)
{
    return lds_bytes(npa, npw, nk, 32, 32, dirs) <= LDS_MAX ? 32 : 16;
}

template <typename T> __device__ __forceinline__ uint32_t ld_raw(win_t w, uint32_t off)
{
    if constexpr (sizeof(T) == 4) return __builtin_amdgcn_raw_buffer_load_b32(w, (int)off, 0, 0);
    return win_load_u16(w, off);
}
template <typename T> __device__ __forceinline__ float raw_float(uint32_t r)
{
    if constexpr (sizeof(T) == 4) {
        return __uint_as_float(r);
    } else {
        T e;
        e.v = (uint16_t)r;
        return Elem<T>::load(&e);
    }
}
template <typename T> __device__ __forceinline__ void st_elem(win_t w, uint32_t off, float v)
{
    if constexpr (sizeof(T) == 4) {
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), w, (int)off, 0, 0);
    } else {
        T e;
        Elem<T>::store(&e, v);
        __builtin_amdgcn_raw_buffer_store_b16(e.v, w, (int)off, 0, 0);
    }
}

// v as N bf16 planes
template <int N> __device__ __forceinline__ void split_planes(float v, uint16_t (&o)[N])
{
#pragma unroll
    for (int m = 0; m < N; ++m) {
        o[m] = (uint16_t)float_to_bf16_bits(v);
        if (m + 1 < N) v -= bf16_bits_to_float(o[m]);
    }
}

__device__ __forceinline__ bf16x8 lds_aligned8(const uint16_t *p)
{
    const uint4 t = *(const uint4 *)p;
    bf16x8 r;
    __builtin_memcpy(&r, &t, 16);
    return r;
}
// 8 consecutive 16-bit elements from an even or odd element index of a 4-byte aligned row (reads two beyond them)
__device__ __forceinline__ bf16x8 lds_any8(const uint16_t *row, int idx)
{
    const uint32_t *p = (const uint32_t *)row + (idx >> 1);
    const uint32_t sh = (uint32_t)(idx & 1) << 4;
    uint32_t d[5], o[4];
#pragma unroll
    for (int i = 0; i < 5; ++i) d[i] = p[i];
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = __builtin_amdgcn_alignbit(d[i + 1], d[i], sh);
    bf16x8 r;
    __builtin_memcpy(&r, o, 16);
    return r;
}
__device__ __forceinline__ bf16x8 negated(bf16x8 v)
{
    uint32_t o[4];
    __builtin_memcpy(o, &v, 16);
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] ^= 0x80008000u;
    __builtin_memcpy(&v, o, 16);
    return v;
}
// plane products a_m b_n with m + n <= 2, smallest first
template <int NA, int NB>
__device__ __forceinline__ f32x4 mfma_planes(const bf16x8 (&a)[NA], const bf16x8 (&b)[NB], f32x4 c)
{
#pragma unroll
    for (int sum = 2; sum >= 0; --sum)
#pragma unroll
        for (int m = 0; m <= sum; ++m)
            if (m < NA && sum - m < NB) c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[m], b[sum - m], c, 0, 0, 0);
    return c;
}

template <int R> __device__ __forceinline__ int wrap(int pos)      // pos in [0, 2 R)
{
    return (int)min((uint32_t)pos, (uint32_t)(pos - R));
}

// 8 samples of channel cl into every plane of a ring at position pos (a multiple of 8)
template <typename T, int NK, int CB>
__device__ __forceinline__ void ring_store(uint16_t *ring, int cl, int pos, const float (&f)[8])
{
    typedef Reach<NK> G;
    constexpr int NPA = GT<T>::NPA;
    uint32_t v[NPA][4];                          // (two samples a conversion: split_planes of each)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        float r0 = f[2 * e] * LIFT<T>, r1 = f[2 * e + 1] * LIFT<T>;
#pragma unroll
        for (int m = 0; m < NPA; ++m) {
            v[m][e] = pack_bf16x2(r0, r1);
            if (m + 1 < NPA) {
                r0 -= __uint_as_float(v[m][e] << 16);
                r1 -= __uint_as_float(v[m][e] & 0xffff0000u);
            }
        }
    }
#pragma unroll
    for (int m = 0; m < NPA; ++m) {
        const uint4 t = make_uint4(v[m][0], v[m][1], v[m][2], v[m][3]);
        uint16_t *row = ring + (m * CB + cl) * G::RP;
        *(uint4 *)(row + pos) = t;
        if (pos == 0) *(uint4 *)(row + G::R) = t;
    }
}

// taps of the workgroup's filters by lag, as planes: tab[plane][filter][z + 16], z = k - m
//   BWD = false: lag = OFF - z (the causal product); true: lag = z (the anti-causal one)
template <typename T, int NK, bool BWD>
__device__ __forceinline__ void fill_taps(uint16_t *tab, const typename Filt<T>::type *h, int64_t f0, int nf, int hl,
                                          int tid, int nt)
{
    typedef Reach<NK> G;
    constexpr int NPW = GT<T>::NPW;
    typedef typename Filt<T>::type FT;
    for (int i = tid; i < nf * G::HP; i += nt) {
        const int f = i / G::HP, z = i - f * G::HP - 16;
        const int lag = BWD ? z : G::OFF - z;
        float v = 0.f;
        if (lag >= 0 && lag < hl) v = Elem<FT>::load(h + (f0 + f) * hl + (hl - 1 - lag));
        uint16_t o[NPW];
        split_planes<NPW>(v * LIFT<FT>, o);
#pragma unroll
        for (int m = 0; m < NPW; ++m) tab[(m * nf + f) * G::HP + z + 16] = o[m];
    }
}

// y[m, n] of the wave's two channels cl0, cl0 + 1 (filters f0, f1 of the table): the NK products of a tile
template <typename T, int NK, int CB>
__device__ __forceinline__ void band_product(f32x4 (&acc)[2], const uint16_t *ring, const uint16_t *tab, int nf, int f0,
                                             int f1, int cl0, int oldest, int lane)
{
    typedef Reach<NK> G;
    constexpr int NPA = GT<T>::NPA, NPW = GT<T>::NPW;
    const int n = lane & 15, q = lane >> 4;
    acc[0] = acc[1] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < NK; ++i) {
        bf16x8 a[NPW], b[NPA];
        const int z = 32 * i + 8 * q + 16 - n;            // (operand row m = n of the lane)
        const int pos = wrap<G::R>(oldest + 16 * n + 32 * i + 8 * q);
#pragma unroll
        for (int m = 0; m < NPW; ++m) a[m] = lds_any8(tab + (m * nf + f0) * G::HP, z);
#pragma unroll
        for (int m = 0; m < NPA; ++m) b[m] = lds_aligned8(ring + (m * CB + cl0) * G::RP + pos);
        acc[0] = mfma_planes(a, b, acc[0]);
        if (f1 != f0)
#pragma unroll
            for (int m = 0; m < NPW; ++m) a[m] = lds_any8(tab + (m * nf + f1) * G::HP, z);
#pragma unroll
        for (int m = 0; m < NPA; ++m) b[m] = lds_aligned8(ring + (m * CB + cl0 + 1) * G::RP + pos);
        acc[1] = mfma_planes(a, b, acc[1]);
    }
}

__device__ __forceinline__ bool all_finite(const float (&v)[8])
{
    float z = 0.f;                               // NaN from the first value on that is not
#pragma unroll
    for (int e = 0; e < 8; ++e) z = fmaf(v[e], 0.f, z);
    return z == 0.f;
}
// a[t] b[t] of one channel (rows ra, rb elements apart), zero outside the sequence
template <typename T>
__device__ __forceinline__ float product_at(const T *a, const T *b, int64_t ra, int64_t rb, int64_t t, int64_t L)
{
    return t >= 0 && t < L ? Elem<T>::load(a + t * ra) * Elem<T>::load(b + t * rb) : 0.f;
}
// one row of a channel: sum over lags of h[lag] times the sample DIR * lag rows on
template <typename FT, int CB, int DIR> __device__ __forceinline__ float row_by_tap(const float *at, const FT *taps, int hl)
{
    float v = 0.f;
#pragma unroll 1
    for (int lag = 0; lag < hl; ++lag) v = fmaf(Elem<FT>::load(taps + (hl - 1 - lag)), at[DIR * lag * CB], v);
    return v;
}

struct Plan {
    int nct, ntile, nseg, tps, nf;               // channel blocks, tiles of a row, runs, tiles per run, filters per block
    int64_t rows, b0;                            // batch rows of a launch, and its first
    int64_t nwg;                                 // workgroups of a launch
};

// where a workgroup is: channel block fastest, then run, then batch row, contiguous per XCD so that the
// workgroups sharing 128-byte lines share an L2
struct Place { int ct, seg; int64_t b; };
__device__ __forceinline__ Place place(const Plan &p)
{
    uint32_t id = xcd_contiguous_u32(blockIdx.x, gridDim.x);
    Place r;
    r.ct = (int)(id % (uint32_t)p.nct); id /= (uint32_t)p.nct;
    r.seg = (int)(id % (uint32_t)p.nseg);
    r.b = p.b0 + id / (uint32_t)p.nseg;
    return r;
}

template <typename T, int NK, int CB>
__global__ __launch_bounds__(32 * CB) void toep_fwd_kernel(const T *__restrict__ x, const T *__restrict__ B,
                                                           const T *__restrict__ C, const void *__restrict__ h,
                                                           T *__restrict__ y, T *__restrict__ y2, T *__restrict__ bx,
                                                           Dims dm, Plan p)
{
    typedef Reach<NK> G;
    typedef typename Filt<T>::type FT;
    constexpr int NPA = GT<T>::NPA, NT = 32 * CB;
    extern __shared__ __align__(16) unsigned char smem[];
    int *const flag = (int *)smem;                                        // the run has to be done again by taps
    uint16_t *ring = (uint16_t *)(smem + 16);
    float *yt = (float *)(ring + NPA * CB * G::RP);
    uint16_t *tab = (uint16_t *)(yt + CB * YP);

    const Place pl = place(p);
    const int tid = threadIdx.x, cl = tid % CB, tg = tid / CB;            // row layout: channel cl, rows 8 tg .. 8 tg + 7
    const int lane = tid & 63, cw = 2 * (tid >> 6);                       // product layout: channels cw, cw + 1
    const int64_t c0 = (int64_t)pl.ct * CB, d = dm.d;
    const int64_t T0 = (int64_t)pl.seg * p.tps * TT, T1 = min(dm.L, T0 + (int64_t)p.tps * TT);
    const int64_t tw = T0 > G::OFF ? T0 - G::OFF : 0;                     // first row of the windows
    const int64_t rowi = (dm.planar ? 3 : dm.es) * d;                     // elements between rows of x, B, C
    const int64_t base_i = (pl.b * dm.L + tw) * rowi, base_o = (pl.b * dm.L + tw) * d;
    const int64_t nrow = T1 - tw;
    const win_t wx = make_window(x + base_i, nrow * rowi * (int64_t)sizeof(T));
    const win_t wB = make_window(B + base_i, nrow * rowi * (int64_t)sizeof(T));
    const win_t wC = make_window(C + base_i, nrow * rowi * (int64_t)sizeof(T));
    const win_t wy = make_window(y + base_o, nrow * d * (int64_t)sizeof(T));
    const win_t wy2 = make_window(y2 ? y2 + base_o : y, y2 ? nrow * d * (int64_t)sizeof(T) : 0);
    const win_t wbx = make_window(bx ? bx + base_o : y, bx ? nrow * d * (int64_t)sizeof(T) : 0);
    const uint32_t lane_off = c0 + cl < d ? 0u : WIN_OFF;
    const uint32_t ri = (uint32_t)(rowi * sizeof(T)), ro = (uint32_t)(d * sizeof(T));
    const uint32_t ci = (uint32_t)((c0 + cl) * dm.es * sizeof(T)) + lane_off, co = (uint32_t)((c0 + cl) * sizeof(T)) + lane_off;

    const int64_t f0 = c0 / dm.dg;
    const int64_t clast = min(c0 + CB, d) - 1;
    const int nf = (int)(clast / dm.dg - f0) + 1;
    const int fa = (int)(min(c0 + cw, clast) / dm.dg - f0), fb = (int)(min(c0 + cw + 1, clast) / dm.dg - f0);
    if (tid == 0) *flag = 0;
    fill_taps<T, NK, false>(tab, (const FT *)h, f0, nf, dm.hl, tid, NT);

    int oldest = 0;                                                       // ring position of row t0 - OFF
    for (int g = tg; g < G::OFF / 8; g += 32) {                           // history of the first tile
        float u[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const uint32_t off = (uint32_t)(int32_t)(T0 - G::OFF - tw + 8 * g + e) * ri + ci;
            u[e] = raw_float<T>(ld_raw<T>(wx, off)) * raw_float<T>(ld_raw<T>(wB, off));
        }
        ring_store<T, NK, CB>(ring, cl, 8 * g, u);
    }
    uint32_t rx[8], rB[8], rC[8];
    // offsets of the thread's first row, running (as products each access costs a multiplication at a quarter of the rate)
    uint32_t oi = ((uint32_t)(T0 - tw) + 8 * tg) * ri + ci, oo = ((uint32_t)(T0 - tw) + 8 * tg) * ro + co;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const uint32_t off = oi + e * ri;
        rx[e] = ld_raw<T>(wx, off); rB[e] = ld_raw<T>(wB, off); rC[e] = ld_raw<T>(wC, off);
    }
    for (int64_t t0 = T0; t0 < T1; t0 += TT, oi += TT * ri, oo += TT * ro) {
        float u[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) u[e] = raw_float<T>(rx[e]) * raw_float<T>(rB[e]);
        ring_store<T, NK, CB>(ring, cl, wrap<G::R>(oldest + G::OFF + 8 * tg), u);
        if (bx)
#pragma unroll
            for (int e = 0; e < 8; ++e) st_elem<T>(wbx, oo + e * ro, u[e]);
        __syncthreads();
#pragma unroll
        for (int e = 0; e < 8; ++e) {                                     // next tile; past the run the window ends
            const uint32_t off = oi + (TT + e) * ri;
            rx[e] = ld_raw<T>(wx, off); rB[e] = ld_raw<T>(wB, off);
        }
        f32x4 acc[2];
        band_product<T, NK, CB>(acc, ring, tab, nf, fa, fb, cw, oldest, lane);
        *(f32x4 *)(yt + cw * YP + 16 * (lane & 15) + 4 * (lane >> 4)) = acc[0] * DROP<T>;
        *(f32x4 *)(yt + (cw + 1) * YP + 16 * (lane & 15) + 4 * (lane >> 4)) = acc[1] * DROP<T>;
        __syncthreads();
        float v[8];
        *(f32x4 *)v = *(const f32x4 *)(yt + cl * YP + 8 * tg);
        *(f32x4 *)(v + 4) = *(const f32x4 *)(yt + cl * YP + 8 * tg + 4);
        if (!all_finite(v)) *flag = 1;
        if (y2)
#pragma unroll
            for (int e = 0; e < 8; ++e) st_elem<T>(wy2, oo + e * ro, v[e]);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float cv = raw_float<T>(rC[e]);
            rC[e] = ld_raw<T>(wC, oi + (TT + e) * ri);
            st_elem<T>(wy, oo + e * ro, cv * v[e]);
        }
        oldest = wrap<G::R>(oldest + TT);
    }
    __syncthreads();
    if (*flag == 0) return;
    // the run again by taps, each row by the thread that stored it: u of a tile and its reach as fp32, rows of CB
    // (the index is hidden from the compiler: what follows from it shall not take registers of the loop above)
    int again = tid;
    asm volatile("" : "+v"(again));
    const int cr = again % CB, tr = again / CB;
    float *const us = (float *)ring;
    const int64_t c = min(c0 + cr, clast), in0 = pl.b * dm.L * rowi + c * dm.es, out0 = pl.b * dm.L * d + c;
    const FT *const taps = (const FT *)h + (c / dm.dg) * dm.hl;
    for (int64_t t0 = T0; t0 < T1; t0 += TT) {
        __syncthreads();
        for (int r = tr; r < G::R; r += 32) us[r * CB + cr] = product_at<T>(x + in0, B + in0, rowi, rowi, t0 - G::OFF + r, dm.L);
        __syncthreads();
#pragma unroll 1
        for (int r = 8 * tr; r < 8 * tr + 8; ++r) {
            const int64_t t = t0 + r;
            if (t >= T1 || c0 + cr >= d) break;
            const float v = row_by_tap<FT, CB, -1>(us + (G::OFF + r) * CB + cr, taps, dm.hl);
            if (y2) Elem<T>::store(y2 + out0 + t * d, v);
            Elem<T>::store(y + out0 + t * d, Elem<T>::load(C + in0 + t * rowi) * v);
        }
    }
}

template <typename T, int NK, int CB>
__global__ __launch_bounds__(32 * CB) void toep_bwd_kernel(const T *__restrict__ dy, const T *__restrict__ x,
                                                           const T *__restrict__ B, const T *__restrict__ C,
                                                           const void *__restrict__ h, T *__restrict__ dx,
                                                           T *__restrict__ dB, T *__restrict__ dC,
                                                           float *__restrict__ ws, Dims dm, Plan p)
{
    typedef Reach<NK> G;
    typedef typename Filt<T>::type FT;
    constexpr int NPA = GT<T>::NPA, NPW = GT<T>::NPW, NT = 32 * CB;
    extern __shared__ __align__(16) unsigned char smem[];
    int *const flag = (int *)smem;
    uint16_t *ru = (uint16_t *)(smem + 16), *rg = ru + NPA * CB * G::RP;
    float *yt = (float *)(rg + NPA * CB * G::RP);
    uint16_t *ta = (uint16_t *)(yt + CB * YP);

    const Place pl = place(p);
    const int tid = threadIdx.x, cl = tid % CB, tg = tid / CB;
    const int lane = tid & 63, cw = 2 * (tid >> 6);
    const int64_t c0 = (int64_t)pl.ct * CB, d = dm.d;
    const int64_t T0 = (int64_t)pl.seg * p.tps * TT, T1 = min(dm.L, T0 + (int64_t)p.tps * TT);
    const int64_t tw = T0 > G::OFF ? T0 - G::OFF : 0, te = min(dm.L, T1 + G::OFF);
    const int64_t rowi = (dm.planar ? 3 : dm.es) * d;
    const int64_t base_i = (pl.b * dm.L + tw) * rowi, base_o = (pl.b * dm.L + tw) * d;
    // x, B and the gradients end with the run, dy and C with its look-ahead
    const int64_t nbi = (T1 - tw) * rowi * (int64_t)sizeof(T);
    const win_t wx = make_window(x + base_i, nbi), wB = make_window(B + base_i, nbi);
    const win_t wC = make_window(C + base_i, (te - tw) * rowi * (int64_t)sizeof(T));
    const win_t wdy = make_window(dy + base_o, (te - tw) * d * (int64_t)sizeof(T));
    const win_t wdx = make_window(dx + base_i, nbi), wdB = make_window(dB + base_i, nbi), wdC = make_window(dC + base_i, nbi);
    const uint32_t lane_off = c0 + cl < d ? 0u : WIN_OFF;
    const uint32_t ri = (uint32_t)(rowi * sizeof(T)), ro = (uint32_t)(d * sizeof(T));
    const uint32_t ci = (uint32_t)((c0 + cl) * dm.es * sizeof(T)) + lane_off, co = (uint32_t)((c0 + cl) * sizeof(T)) + lane_off;

    const int64_t f0 = c0 / dm.dg;
    const int64_t clast = min(c0 + CB, d) - 1;
    const int nf = (int)(clast / dm.dg - f0) + 1;
    const int fa = (int)(min(c0 + cw, clast) / dm.dg - f0), fb = (int)(min(c0 + cw + 1, clast) / dm.dg - f0);
    uint16_t *tb = ta + NPW * nf * G::HP;
    if (tid == 0) *flag = 0;
    fill_taps<T, NK, false>(ta, (const FT *)h, f0, nf, dm.hl, tid, NT);
    fill_taps<T, NK, true>(tb, (const FT *)h, f0, nf, dm.hl, tid, NT);

    int oldest = 0, front = 0;                                            // ring positions of u[t0 - OFF] and g2[t0]
    for (int g = tg; g < G::OFF / 8; g += 32) {
        float u[8], v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const uint32_t off = (uint32_t)(int32_t)(T0 - G::OFF - tw + 8 * g + e) * ri + ci;
            u[e] = raw_float<T>(ld_raw<T>(wx, off)) * raw_float<T>(ld_raw<T>(wB, off));
        }
        ring_store<T, NK, CB>(ru, cl, 8 * g, u);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const uint32_t r = (uint32_t)(T0 - tw) + 8 * g + e;
            v[e] = raw_float<T>(ld_raw<T>(wdy, r * ro + co)) * raw_float<T>(ld_raw<T>(wC, r * ri + ci));
        }
        ring_store<T, NK, CB>(rg, cl, 8 * g, v);
    }
    uint32_t rx[8], rB[8], rl[8], rC[8], rd[8];                           // rl, rC: dy and C of the look-ahead; rd: dy of the tile
    uint32_t oi = ((uint32_t)(T0 - tw) + 8 * tg) * ri + ci, oo = ((uint32_t)(T0 - tw) + 8 * tg) * ro + co;   // (running: see the forward)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        rx[e] = ld_raw<T>(wx, oi + e * ri); rB[e] = ld_raw<T>(wB, oi + e * ri);
        rl[e] = ld_raw<T>(wdy, oo + (G::OFF + e) * ro); rC[e] = ld_raw<T>(wC, oi + (G::OFF + e) * ri);
    }
    f32x4 dh[2];
    dh[0] = dh[1] = (f32x4){0.f, 0.f, 0.f, 0.f};
    const int n = lane & 15, q = lane >> 4;
    const int ga = min(n, (dm.hl - 1) >> 4) * 16;                         // row a of the filter-gradient tile, in samples
    for (int64_t t0 = T0; t0 < T1; t0 += TT, oi += TT * ri, oo += TT * ro) {
        float u[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) u[e] = raw_float<T>(rx[e]) * raw_float<T>(rB[e]);
        ring_store<T, NK, CB>(ru, cl, wrap<G::R>(oldest + G::OFF + 8 * tg), u);
#pragma unroll
        for (int e = 0; e < 8; ++e) u[e] = raw_float<T>(rl[e]) * raw_float<T>(rC[e]);
        ring_store<T, NK, CB>(rg, cl, wrap<G::R>(front + G::OFF + 8 * tg), u);
        __syncthreads();
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            rd[e] = ld_raw<T>(wdy, oo + e * ro);
            rl[e] = ld_raw<T>(wdy, oo + (TT + G::OFF + e) * ro); rC[e] = ld_raw<T>(wC, oi + (TT + G::OFF + e) * ri);
        }
        f32x4 acc[2];
        float v[8];
        float *const yw = yt + cw * YP + 16 * n + 4 * q, *const yr = yt + cl * YP + 8 * tg;
        band_product<T, NK, CB>(acc, ru, ta, nf, fa, fb, cw, oldest, lane);
        *(f32x4 *)yw = acc[0] * DROP<T>;
        *(f32x4 *)(yw + YP) = acc[1] * DROP<T>;
        __syncthreads();
        *(f32x4 *)v = *(const f32x4 *)yr;
        *(f32x4 *)(v + 4) = *(const f32x4 *)(yr + 4);
#pragma unroll
        for (int e = 0; e < 8; ++e) st_elem<T>(wdC, oi + e * ri, raw_float<T>(rd[e]) * v[e]);
        if (!all_finite(v)) *flag = 1;
        // filter gradient: 32 rows' products by themselves, added to the tile's sum and that to the run's; half of the
        // products with a negated operand (see the head of this file)
        f32x4 dt[2];
        dt[0] = dt[1] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int neg = 0; neg < 2; ++neg)
#pragma unroll 1
            for (int s = neg * (TT / 64); s < (neg + 1) * (TT / 64); ++s) {
                const int pg = wrap<G::R>(front + 32 * s + 8 * q + ga), pu = wrap<G::R>(oldest + G::OFF + 32 * s + 8 * q - n);
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    bf16x8 a[NPA], b[NPA];
#pragma unroll
                    for (int m = 0; m < NPA; ++m) {
                        a[m] = lds_aligned8(rg + (m * CB + cw + c) * G::RP + pg);
                        if (neg) a[m] = negated(a[m]);
                        b[m] = lds_any8(ru + (m * CB + cw + c) * G::RP, pu);
                    }
                    const f32x4 t = mfma_planes(a, b, (f32x4){0.f, 0.f, 0.f, 0.f});
                    dt[c] = neg ? dt[c] - t : dt[c] + t;
                }
            }
        dh[0] += dt[0];
        dh[1] += dt[1];
        band_product<T, NK, CB>(acc, rg, tb, nf, fa, fb, cw, front, lane);
        __syncthreads();
        *(f32x4 *)yw = acc[0] * DROP<T>;
        *(f32x4 *)(yw + YP) = acc[1] * DROP<T>;
        __syncthreads();
        *(f32x4 *)v = *(const f32x4 *)yr;
        *(f32x4 *)(v + 4) = *(const f32x4 *)(yr + 4);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const uint32_t o = oi + e * ri;
            const float xv = raw_float<T>(rx[e]), bv = raw_float<T>(rB[e]);
            rx[e] = ld_raw<T>(wx, o + TT * ri); rB[e] = ld_raw<T>(wB, o + TT * ri);
            st_elem<T>(wdx, o, v[e] * bv);
            st_elem<T>(wdB, o, v[e] * xv);
        }
        if (!all_finite(v)) *flag = 1;
        oldest = wrap<G::R>(oldest + TT);
        front = wrap<G::R>(front + TT);
    }
    // this run's filter gradient by lag: the channels of a filter added in their order
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (!(dh[c][r] * 0.f == 0.f)) *flag = 1;                      // (2^48 times the sum: past the range earlier)
    __syncthreads();
    if (*flag == 0) {
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int r = 0; r < 4; ++r) yt[(cw + c) * TT + (4 * q + r) * 16 + n] = dh[c][r] * (1.f / (LIFT<T> * LIFT<T>));
    } else {
        // the run again by taps, each row by the thread that stored it and lags tr, tr + 32, ... of its channel: u and g2
        // of a tile and their reach as fp32, rows of CB
        int again = tid;
        asm volatile("" : "+v"(again));
        const int cr = again % CB, tr = again / CB;
        float *const us = (float *)ru, *const gs = (float *)rg;
        const int64_t c = min(c0 + cr, clast), in0 = pl.b * dm.L * rowi + c * dm.es, out0 = pl.b * dm.L * d + c;
        const FT *const taps = (const FT *)h + (c / dm.dg) * dm.hl;
        for (int lag = tr; lag < dm.hl; lag += 32) yt[cr * TT + lag] = 0.f;
        for (int64_t t0 = T0; t0 < T1; t0 += TT) {
            __syncthreads();
            for (int r = tr; r < G::R; r += 32) {
                us[r * CB + cr] = product_at<T>(x + in0, B + in0, rowi, rowi, t0 - G::OFF + r, dm.L);
                gs[r * CB + cr] = product_at<T>(dy + out0, C + in0, d, rowi, t0 + r, dm.L);
            }
            __syncthreads();
#pragma unroll 1
            for (int r = 8 * tr; r < 8 * tr + 8; ++r) {
                const int64_t t = t0 + r, o = in0 + t * rowi;
                if (t >= T1 || c0 + cr >= d) break;
                Elem<T>::store(dC + o, Elem<T>::load(dy + out0 + t * d) *
                                           row_by_tap<FT, CB, -1>(us + (G::OFF + r) * CB + cr, taps, dm.hl));
                const float du = row_by_tap<FT, CB, 1>(gs + r * CB + cr, taps, dm.hl);
                Elem<T>::store(dx + o, du * Elem<T>::load(B + o));
                Elem<T>::store(dB + o, du * Elem<T>::load(x + o));
            }
#pragma unroll 1
            for (int lag = tr; lag < dm.hl; lag += 32) {
                const int a = lag & ~15, b = lag & 15;                     // as the products cut it: g2[s + a] u[s - b]
                float s = yt[cr * TT + lag];
#pragma unroll 1
                for (int r = 0; r < TT; ++r)
                    if (t0 + r + a < dm.L && t0 + r - b >= 0) s = fmaf(gs[(r + a) * CB + cr], us[(G::OFF + r - b) * CB + cr], s);
                yt[cr * TT + lag] = s;
            }
        }
    }
    __syncthreads();
    float *const slot = ws + (size_t)(((pl.b - p.b0) * p.nseg + pl.seg) * p.nct + pl.ct) * p.nf * dm.hl;
    for (int i = tid; i < nf * dm.hl; i += NT) {
        const int f = i / dm.hl, k = i - f * dm.hl;
        const int64_t lo = (f0 + f) * dm.dg - c0, hi = lo + dm.dg;
        const int a = (int)max((int64_t)0, lo), b = (int)min(hi, clast + 1 - c0);
        float s = 0.f;
        for (int c = a; c < b; ++c) s += yt[c * TT + dm.hl - 1 - k];
        slot[i] = p.b0 ? slot[i] + s : s;
    }
}

// dh[grp, k] = sum over the batch rows of a launch, runs and the channel blocks that touch the group, in that order
template <typename FT>
__global__ __launch_bounds__(64) void toep_dh_kernel(const float *__restrict__ ws, FT *__restrict__ dh, Dims dm, Plan p,
                                                     int cb)
{
    const int64_t i = (int64_t)blockIdx.x * 64 + threadIdx.x;
    if (i >= (int64_t)dm.g * dm.hl) return;
    const int64_t grp = i / dm.hl, k = i - grp * dm.hl;
    const int64_t lo = grp * dm.dg / cb, hi = ((grp + 1) * dm.dg - 1) / cb;
    float s = 0.f;
    for (int64_t ct = lo; ct <= hi; ++ct) {
        const int64_t f = grp - ct * cb / dm.dg;
        const float *w = ws + (ct * p.nf + f) * dm.hl + k;
        const int64_t step = (int64_t)p.nct * p.nf * dm.hl, n = p.rows * p.nseg;
        int64_t r = 0;
        for (; r + 8 <= n; r += 8) {
            float v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = w[(r + e) * step];
#pragma unroll
            for (int e = 0; e < 8; ++e) s += v[e];
        }
        for (; r < n; ++r) s += w[r * step];
    }
    Elem<FT>::store(dh + i, s);
}

int pick_nk(int hl) { return hl <= 17 ? 1 : hl <= 81 ? 3 : hl <= 145 ? 5 : 9; }
int npa_of(int dtype) { return dtype == GCG_BF16 || dtype == GCG_BF16_F32 ? 2 : 3; }
int npw_of(int dtype) { return dtype == GCG_BF16 ? 1 : dtype == GCG_F16 ? 2 : 3; }

// Tiles per run, at most cap: as many runs as make rounds of one workgroup per CU x (tiles of a run + the reach it loads
// first) smallest.  For a number of rounds the best run is the shortest that needs no more; no more rounds are tried once
// their leads alone, on top of the work spread evenly, cost what the best cut does (two or three as a rule: the query that
// sizes a backward's workspace comes through here on every call).
int pick_tps(int64_t cols, int64_t ntile, int64_t cap, int64_t cus, int lead)
{
    const int64_t fewest = (ntile + cap - 1) / cap, least = cols * ntile * TT / cus;
    int64_t rounds = (cols * fewest + cus - 1) / cus, best = INT64_MAX, tps = cap;
    for (int64_t tries = 0; tries < 64 && least + rounds * lead < best; ++tries, ++rounds) {
        int64_t runs = rounds * cus / cols;
        if (runs > ntile) runs = ntile;
        const int64_t n = (ntile + runs - 1) / runs, cost = rounds * (n * TT + lead);
        if (cost < best) { best = cost; tps = n; }
    }
    return (int)tps;
}

// vector_bytes: what the vector kernels' backward of these sizes keeps partial sums in.  False: sizes for those kernels.
bool make_plan(int dtype, const Dims &dm, int dirs, size_t vector_bytes, Plan &p)
{
    if (dm.hl < 9 || dm.hl > 256 || dm.tmajor) return false;
    const int npa = npa_of(dtype), npw = npw_of(dtype), nk = pick_nk(dm.hl), cb = pick_cb(npa, npw, nk, dirs);
    p.nct = (int)((dm.d + cb - 1) / cb);
    p.ntile = (int)((dm.L + TT - 1) / TT);
    p.nf = (int)((cb - 1) / dm.dg + 2 < cb ? (cb - 1) / dm.dg + 2 : cb);
    if (cb % dm.dg == 0) p.nf = cb / dm.dg;
    else if (dm.dg % cb == 0) p.nf = 1;
    if (lds_bytes(npa, npw, nk, cb, p.nf, dirs) > LDS_MAX) return false;
    const int64_t cols = dm.bs * p.nct;
    // rows of a run: what a window spans (with the reach on both sides; the workspace query does not know the layout,
    // so always that of a features tensor), no more tiles than there are, and 256: the tiles' sums of the filter gradient
    // are added one after the other (a run's lead is 0.3 % of that)
    const int64_t esz = dtype == GCG_F32 ? 4 : 2, rowb = 3 * dm.d * esz;
    int64_t cap = (WIN_MAX_BYTES / rowb - 2 * (32 * nk - 16)) / TT;
    if (cap > p.ntile) cap = p.ntile;
    if (cap > 256) cap = 256;
    if (cap <= 0) return false;
    const int lead = dirs * (32 * nk - 16) / 2 + 64;
    p.tps = pick_tps(cols, p.ntile, cap, cu_count(), lead);
    p.nseg = (p.ntile + p.tps - 1) / p.tps;
    p.rows = dm.bs;
    p.b0 = 0;
    // A backward whose partial sums the static scratch held with the vector kernels' blocks of 64 channels and does not
    // with these of 16 or 32 is launched for a part of the batch rows at a time, each launch adding to the sums of the
    // one before, here and with a workspace alike (21 x 160 x (256 groups of 32), 256 taps, bf16: 10.5 MB and 587 us in
    // one launch, 5.5 MB and 594 us in two).
    const size_t row_bytes = (size_t)p.nct * p.nseg * p.nf * dm.hl * sizeof(float);
    if (dirs == 2 && vector_bytes <= GCG_BWD_STATIC_SCRATCH_BYTES && dm.bs * row_bytes > GCG_BWD_STATIC_SCRATCH_BYTES) {
        const int64_t rows = (int64_t)(GCG_BWD_STATIC_SCRATCH_BYTES / row_bytes);
        if (rows == 0) return false;
        const int64_t launches = (dm.bs + rows - 1) / rows;
        p.rows = (dm.bs + launches - 1) / launches;
    }
    p.nwg = p.rows * p.nct * p.nseg;
    return p.nwg * 32 * cb <= 0xffffffffLL;      // work-items of a launch
}

template <typename T, int NK>
int fwd_nk(const void *x, const void *B, const void *C, const void *h, void *y, void *y2, void *bx, const Dims &dm,
           const Plan &p, hipStream_t st)
{
    constexpr int CB = pick_cb(GT<T>::NPA, GT<T>::NPW, NK, 1);
    return launch_main_lds(toep_fwd_kernel<T, NK, CB>, dim3((unsigned)p.nwg), dim3(32 * CB),
                           lds_bytes(GT<T>::NPA, GT<T>::NPW, NK, CB, p.nf, 1), st, take_kernel_timer(), (const T *)x,
                           (const T *)B, (const T *)C, h, (T *)y, (T *)y2, (T *)bx, dm, p);
}

template <typename T, int NK>
int bwd_nk(const void *dy, const void *x, const void *B, const void *C, const void *h, void *dx, void *dB, void *dC,
           void *dh, void *ws, const Dims &dm, const Plan &p, hipStream_t st)
{
    constexpr int CB = pick_cb(GT<T>::NPA, GT<T>::NPW, NK, 2);
    typedef typename Filt<T>::type FT;
    const KernelTimer timer = take_kernel_timer();
    for (Plan q = p; q.b0 < dm.bs; q.b0 += q.rows) {
        const int64_t nwg = p.nwg / p.rows * min(p.rows, dm.bs - q.b0);
        const KernelTimer t = {q.b0 ? nullptr : timer.start, q.b0 + q.rows < dm.bs ? nullptr : timer.stop};
        const int e = launch_main_lds(toep_bwd_kernel<T, NK, CB>, dim3((unsigned)nwg), dim3(32 * CB),
                                      lds_bytes(GT<T>::NPA, GT<T>::NPW, NK, CB, p.nf, 2), st, t, (const T *)dy, (const T *)x,
                                      (const T *)B, (const T *)C, h, (T *)dx, (T *)dB, (T *)dC, (float *)ws, dm, q);
        if (e) return e;
    }
    const int64_t n = (int64_t)dm.g * dm.hl;
    return launch_plain(toep_dh_kernel<FT>, dim3((unsigned)((n + 63) / 64)), dim3(64), st, (const float *)ws, (FT *)dh, dm, p,
                        CB);
}

template <typename T, typename... A> int fwd_t(int hl, A... a)
{
    switch (pick_nk(hl)) {
    case 1: return fwd_nk<T, 1>(a...);
    case 3: return fwd_nk<T, 3>(a...);
    case 5: return fwd_nk<T, 5>(a...);
    }
    return fwd_nk<T, 9>(a...);
}
template <typename T, typename... A> int bwd_t(int hl, A... a)
{
    switch (pick_nk(hl)) {
    case 1: return bwd_nk<T, 1>(a...);
    case 3: return bwd_nk<T, 3>(a...);
    case 5: return bwd_nk<T, 5>(a...);
    }
    return bwd_nk<T, 9>(a...);
}

} // namespace

int toep_fwd_launch(int dtype, const void *x, const void *B, const void *C, const void *h, void *y, void *y2, void *bx,
                    const Dims &dm, hipStream_t st)
{
    Plan p;
    if (!make_plan(dtype, dm, 1, 0, p)) return TOEP_NOT_TAKEN;
    switch (dtype) {
    case GCG_F32:  return fwd_t<float>(dm.hl, x, B, C, h, y, y2, bx, dm, p, st);
    case GCG_BF16: return fwd_t<bf16_t>(dm.hl, x, B, C, h, y, y2, bx, dm, p, st);
    case GCG_F16:  return fwd_t<f16_t>(dm.hl, x, B, C, h, y, y2, bx, dm, p, st);
    case GCG_BF16_F32: return fwd_t<bf16w_t>(dm.hl, x, B, C, h, y, y2, bx, dm, p, st);
    case GCG_F16_F32:  return fwd_t<f16w_t>(dm.hl, x, B, C, h, y, y2, bx, dm, p, st);
    }
    return (int)hipErrorInvalidValue;
}

size_t toep_bwd_workspace(int dtype, const Dims &dm, size_t vector_bytes)
{
    Plan p;
    return make_plan(dtype, dm, 2, vector_bytes, p) ? (size_t)p.nwg * p.nf * dm.hl * sizeof(float) : 0;
}

int toep_bwd_launch(int dtype, const void *dy, const void *x, const void *B, const void *C, const void *h, void *dx,
                    void *dB, void *dC, void *dh, void *ws, const Dims &dm, size_t vector_bytes, hipStream_t st)
{
    Plan p;
    if (!make_plan(dtype, dm, 2, vector_bytes, p)) return TOEP_NOT_TAKEN;
    switch (dtype) {
    case GCG_F32:  return bwd_t<float>(dm.hl, dy, x, B, C, h, dx, dB, dC, dh, ws, dm, p, st);
    case GCG_BF16: return bwd_t<bf16_t>(dm.hl, dy, x, B, C, h, dx, dB, dC, dh, ws, dm, p, st);
    case GCG_F16:  return bwd_t<f16_t>(dm.hl, dy, x, B, C, h, dx, dB, dC, dh, ws, dm, p, st);
    case GCG_BF16_F32: return bwd_t<bf16w_t>(dm.hl, dy, x, B, C, h, dx, dB, dC, dh, ws, dm, p, st);
    case GCG_F16_F32:  return bwd_t<f16w_t>(dm.hl, dy, x, B, C, h, dx, dB, dC, dh, ws, dm, p, st);
    }
    return (int)hipErrorInvalidValue;
}

} // namespace gcg
