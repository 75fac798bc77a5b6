// Tall complex-FP64 products for gfx950:
//   * coef_gemm: out[p][l] = alpha * sum_q coef(q,p) * in[q][l] -- the forcing
//     synthesis of SourceCode/CreateForcingOnFly.c:17-19 batched over a chunk
//     of half-step samples and over all k test vectors, the snapshot DFT of
//     SourceCode/DFT.c:26-38, and the windowed DFTs of SourceCode/GalerkinProj.c:30-46.
//     L (= N*k complex columns) is huge and K, P <= ~130, so every workgroup
//     streams a slab of `in` once and keeps a P-tile of accumulators per lane;
//     the coefficient tile is wave-uniform and is read through the scalar cache.
//   * bgram: batched conj(X)^T Z over tall row ranges (Gram matrices of
//     CholeskyQR, the projections V^H(.) of the transient removal), reduced
//     deterministically in two passes.
//   * bapply: batched row-local small products Out = alpha*Y + X*C (the
//     triangular applies of CholeskyQR, Q*U of the SVD, y1 - V*a).
#include "common.h"
#include <type_traits>

namespace rsvdt {

// ----------------------------------------------------------------- coef_gemm
// FP64 MFMA (v_mfma_f64_16x16x4f64).  A wave owns a strip of 16 columns l and
// computes all T*16 rows p of the workgroup's row range for it; the complex
// product is four real MFMAs per K-step of 4:
//   Re += Cr*Xr + (-Ci)*Xi,   Im += Cr*Xi + Ci*Xr.
// Operand layouts (16x16x4, wave64): A(16x4): lane i -> A[i%16][i/16],
// B(4x16): lane i -> B[i/16][i%16], D(16x16): lane i holds D[4j+i/16][i%16], j < 4
// (checked on gfx950 with a known-answer product).
// The K x T*16 coefficient block of the workgroup is staged in LDS once and
// reused for every 64-column tile the workgroup visits (grid-stride), so
// `in` is streamed from HBM exactly once per row range.
typedef double dvec4 __attribute__((ext_vector_type(4)));
typedef double dvec2 __attribute__((ext_vector_type(2)));

// The wave's index in its workgroup, as a scalar: loops and branches on it stay
// uniform for the compiler.
__device__ __forceinline__ int wave_id() { return __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6); }

template <int T, typename OV>
__global__ __launch_bounds__(256) void k_coef_gemm(
    int64_t P, int64_t K, int64_t L, const double2 *__restrict__ coef, int64_t cq, int64_t cp, int64_t p0,
    int sgn, int64_t cmod, double alpha, const double2 *__restrict__ in, int64_t ldi, OV *__restrict__ out,
    int64_t ldo, double beta)
{
    extern __shared__ double2 cs[];                 // [Kpad][T*16 + 4]
    constexpr int PW = T * 16;
    constexpr int PS = PW + 4;                      // row pitch: the 4 rows a K-step reads hit different banks
    const int lane = threadIdx.x & 63, wv = wave_id();
    const int64_t pbase = (int64_t)blockIdx.y * PW;
    const int64_t Kpad = (K + 3) & ~(int64_t)3;
    for (int64_t e = threadIdx.x; e < Kpad * PW; e += 256) {
        const int64_t q = e / PW, pp = e % PW, p = pbase + pp;
        double2 v = make_double2(0, 0);
        if (q < K && p < P) {
            int64_t col = p0 + (int64_t)sgn * p;
            if (col < 0 || col >= cmod) { col %= cmod; if (col < 0) col += cmod; }
            v = coef[q * cq + col * cp];
        }
        cs[q * PS + pp] = v;
    }
    __syncthreads();
    const int kq = lane >> 4, cl = lane & 15;
    const int64_t ntile = (L + 63) / 64;
    // The workgroup's (tile, K-step) sequence is walked as one stream with the
    // streamed operand loaded PF steps ahead, across tile boundaries too; both
    // ends of the stream count steps and move pointers (finding a step's tile by
    // 64-bit division cost more vector instructions than all the rest).  Bound
    // by the FP64 matrix cores: the 64 x 64 x 6.3M forcing chunk takes 3.6 to 3.8 ms
    // (4.2 ms with divisions), 75 to 81 % of their cycles at the 2.05 GHz that this
    // load runs at; PF = 8, 12, 16: 3.87, 3.78, 3.82 ms.
    constexpr int PF = 12;
    const int nks = (int)(Kpad >> 2);
    const int64_t nmine = blockIdx.x < ntile ? (ntile - 1 - blockIdx.x) / gridDim.x + 1 : 0;
    const int64_t nsteps = nmine * nks, hop = (int64_t)gridDim.x * 64;
    int64_t lo = (int64_t)blockIdx.x * 64 + wv * 16 + cl, ll = lo, lleft = nsteps;
    int lks = 0, ks = 0;
    const double2 *lp = in + (kq < K ? kq : 0) * ldi;
    auto load_step = [&]() -> double2 {
        double2 v = make_double2(0, 0);
        if (lleft > 0) {
            if (ll < L && lks * 4 + kq < K) v = lp[ll];
            --lleft;
            lp += 4 * ldi;
            if (++lks == nks) { lks = 0; ll += hop; lp = in + (kq < K ? kq : 0) * ldi; }
        }
        return v;
    };
    double2 ring[PF];
#pragma unroll
    for (int p = 0; p < PF; ++p) ring[p] = load_step();
    dvec4 ar[T], ai[T];
#pragma unroll
    for (int t = 0; t < T; ++t) { ar[t] = (dvec4){0, 0, 0, 0}; ai[t] = (dvec4){0, 0, 0, 0}; }
    for (int64_t g0 = 0; g0 < nsteps; g0 += PF) {
#pragma unroll
        for (int p = 0; p < PF; ++p) {
            if (g0 + p < nsteps) {
                const double2 x = ring[p];
                ring[p] = load_step();
                const double2 *crow = cs + ((int64_t)ks * 4 + kq) * PS + cl;
                double2 c[T];
#pragma unroll
                for (int t = 0; t < T; ++t) c[t] = crow[t * 16];
                // 2T independent accumulators between dependent MFMAs
#pragma unroll
                for (int t = 0; t < T; ++t) {
                    ar[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(c[t].x, x.x, ar[t], 0, 0, 0);
                    ai[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(c[t].x, x.y, ai[t], 0, 0, 0);
                }
#pragma unroll
                for (int t = 0; t < T; ++t) {
                    ar[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(-c[t].y, x.y, ar[t], 0, 0, 0);
                    ai[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(c[t].y, x.x, ai[t], 0, 0, 0);
                }
                if (++ks == nks) {                    // tile done: store and restart the sums
                    ks = 0;
                    const int64_t l = lo;
                    lo += hop;
                    if (l < L) {
#pragma unroll
                        for (int t = 0; t < T; ++t)
#pragma unroll
                            for (int j = 0; j < 4; ++j) {
                                const int64_t pp = pbase + t * 16 + 4 * j + kq;
                                if (pp < P) {
                                    OV *o = out + pp * ldo + l;
                                    double orr = alpha * ar[t][j], oi = alpha * ai[t][j];
                                    if (beta != 0.0) { OV v = *o; orr += beta * (double)v.x; oi += beta * (double)v.y; }
                                    OV w;
                                    w.x = orr; w.y = oi;
                                    *o = w;
                                }
                            }
                    }
#pragma unroll
                    for (int t = 0; t < T; ++t) { ar[t] = (dvec4){0, 0, 0, 0}; ai[t] = (dvec4){0, 0, 0, 0}; }
                }
            }
        }
    }
}

template <int T>
static int launch_coef(int64_t P, int64_t K, int64_t L, const double *coef, int64_t cq, int64_t cp, int64_t p0,
                       int sgn, int64_t cmod, double alpha, const double *in, int64_t ldi, void *out, int64_t ldo,
                       int out_prec, double beta, hipStream_t s)
{
    const int64_t Kpad = (K + 3) & ~(int64_t)3;
    const size_t lds = (size_t)Kpad * (T * 16 + 4) * 16;
    const int64_t ntile = (L + 63) / 64;
    // enough workgroups to fill 256 CUs several times; each visits ntile/gx tiles
    const int64_t per_cu = lds > 80 * 1024 ? 1 : (lds > 40 * 1024 ? 2 : 4);
    int64_t gx = 256 * per_cu * 2;
    if (gx > ntile) gx = ntile;
    dim3 grid((unsigned)gx, ceil_div(P, T * 16));
    if (out_prec == 64)
        hipLaunchKernelGGL((k_coef_gemm<T, double2>), grid, dim3(256), lds, s, P, K, L, (const double2 *)coef, cq, cp,
                           p0, sgn, cmod, alpha, (const double2 *)in, ldi, (double2 *)out, ldo, beta);
    else
        hipLaunchKernelGGL((k_coef_gemm<T, float2>), grid, dim3(256), lds, s, P, K, L, (const double2 *)coef, cq, cp,
                           p0, sgn, cmod, alpha, (const double2 *)in, ldi, (float2 *)out, ldo, beta);
    RSVDT_LAUNCH_CHECK("rsvdt_hip_coef_gemm");
    return RSVDT_HIP_OK;
}

// ----------------------------------------------------------------- bgram
#define BG_T 16
__global__ __launch_bounds__(256) void k_bgram_part(
    int64_t nrows, int64_t na, int64_t nc, int64_t chunk, int ntc,
    const double2 *__restrict__ X, int64_t xb, int64_t xr, int64_t xa,
    const double2 *__restrict__ Z, int64_t zb, int64_t zr, int64_t zc, double2 *__restrict__ part)
{
    __shared__ double2 sx[BG_T][BG_T + 1];
    __shared__ double2 sz[BG_T][BG_T + 1];
    const int64_t b = blockIdx.z;
    const int64_t nch = gridDim.x;
    const int tile = blockIdx.y;
    const int64_t a0 = (int64_t)(tile / ntc) * BG_T, c0 = (int64_t)(tile % ntc) * BG_T;
    const int ti = threadIdx.x / BG_T, tj = threadIdx.x % BG_T;
    const int64_t r_begin = (int64_t)blockIdx.x * chunk;
    int64_t r_end = r_begin + chunk;
    if (r_end > nrows) r_end = nrows;
    const double2 *Xb = X + b * xb;
    const double2 *Zb = Z + b * zb;
    double2 acc = make_double2(0, 0);
    for (int64_t r0 = r_begin; r0 < r_end; r0 += BG_T) {
        const int64_t r = r0 + ti;
        const int64_t a = a0 + tj, c = c0 + tj;
        sx[ti][tj] = (r < r_end && a < na) ? Xb[r * xr + a * xa] : make_double2(0, 0);
        sz[ti][tj] = (r < r_end && c < nc) ? Zb[r * zr + c * zc] : make_double2(0, 0);
        __syncthreads();
#pragma unroll
        for (int rr = 0; rr < BG_T; ++rr) {
            const double2 xv = sx[rr][ti], zv = sz[rr][tj];
            acc.x += xv.x * zv.x + xv.y * zv.y;
            acc.y += xv.x * zv.y - xv.y * zv.x;
        }
        __syncthreads();
    }
    const int64_t a = a0 + ti, c = c0 + tj;
    if (a < na && c < nc) part[((b * nch + blockIdx.x) * na + a) * nc + c] = acc;
}

// G_b(a, c) = sum over the nch partial matrices of batch b, in a fixed order:
// 32 entries x 8 slices of the partials per workgroup (and further entries, as
// a launch takes fewer than 2^24 workgroups), the slices' sums combined through
// LDS.  One thread per entry walking all partials was a serial chain of loads
// (165 us for 16 batches of 512 partials of 16 x 16).
// herm: the tiles below the diagonal (and the border row) were not formed and
// are the conjugates of their mirrors; ntile: the 16-wide tiles (columns from
// 16 ntile on are the border).
__global__ __launch_bounds__(256) void k_bgram_reduce(int64_t nch, int na, int nc, int herm, int ntile,
                                                      const double2 *__restrict__ part, double2 *__restrict__ G)
{
    __shared__ double2 sh[8][32];
    const int64_t b = blockIdx.y;
    const int64_t per = (int64_t)na * nc;
    const int sl = threadIdx.x >> 5;
    for (int64_t e0 = (int64_t)blockIdx.x * 32; e0 < per; e0 += (int64_t)gridDim.x * 32) {
        const int64_t e = e0 + (int)(threadIdx.x & 31);
        double2 s = make_double2(0, 0);
        bool mir = false;
        if (e < per) {
            const int a = (int)(e / nc), c = (int)(e % nc);
            const int ta = min(a / 16, ntile), tc = min(c / 16, ntile);
            mir = herm && ta > tc;
            const double2 *p = part + b * nch * per + (mir ? (int64_t)c * nc + a : e);
            for (int64_t ch = sl; ch < nch; ch += 8) {
                const double2 v = p[ch * per];
                s.x += v.x; s.y += v.y;
            }
        }
        sh[sl][threadIdx.x & 31] = s;
        __syncthreads();
        if (sl == 0 && e < per) {
#pragma unroll
            for (int q = 1; q < 8; ++q) { s.x += sh[q][threadIdx.x].x; s.y += sh[q][threadIdx.x].y; }
            G[b * per + e] = make_double2(s.x, mir ? -s.y : s.y);
        }
        __syncthreads();
    }
}

// FP64 MFMA Gram for unit column strides (rows of X and Z contiguous, the
// per-batch row-major layout).  A workgroup forms a (16 TA) x (16 TC) macro
// tile of G = X^H Z over a row chunk, complex as four real products:
//   Re G += Xr Zr + Xi Zi,   Im G += Xr Zi - Xi Zr.
// A(16x4): lane i -> X(r0 + i/16, a0 + i%16); B(4x16): lane i -> Z(r0 + i/16,
// c0 + i%16); D: lane i holds G(a0 + 4j + i/16, c0 + i%16), j < 4.
// The four waves take every fourth 4-row step and the whole macro tile each,
// or, for 4 x 4 tiles (256 accumulator registers would not leave room for the
// operands), every other step and half of the tile's rows (GA = 2).  Their
// sums are combined through LDS in a fixed order and the chunk's partial goes
// to k_bgram_reduce.
// What bounds it: FP64 MFMA for n above 16, memory for one tile.  Hence
//   * BORD: n = 16 T + 1 columns (the Nw + 1 snapshots of a removal) keep T
//     tiles; the one border column and row are plain FMAs on the operands
//     the lanes hold anyway (for n = 65: 16 MFMA tiles instead of 25);
//   * HERM: X and Z the same array (CholeskyQR) forms the upper tiles only;
//   * PF row steps are in flight per wave where the MFMAs of a step do not
//     cover a load's latency; the loads are branch-free (clamped addresses,
//     zeros selected afterwards).
// 8 batches of 98,304 x 65 (V^H X of a removal): 483 us, 55 TFLOP/s (48 x 48
// tiles per wave, padded to 96 x 96: 1620 us).  16 batches of 393,216 x 16
// (QR): 329 us, 4.9 TB/s, with nontemporal loads and 8 steps in flight; 351 us
// without the hint, 377 us with one step in flight.  The launch bound keeps
// two waves per SIMD for half tiles (742 us with one).
template <int TA, int TC, bool HERM, bool BORD>
__global__ __launch_bounds__(256, TA *TC <= 1 ? 4 : (TA == 4 && !HERM ? 2 : 1)) void k_bgram_mfma(
    int64_t nrows, int na, int nc, int64_t chunk, int tile0, int ntc, const double2 *X, int64_t xb, int64_t xr,
    const double2 *Z, int64_t zb, int64_t zr, double2 *__restrict__ part)
{
    constexpr int GA = TA == 4 && !HERM ? 2 : 1, WA = TA / GA, NSUB = 4 / GA;
    constexpr int PF = TA * TC == 1 ? (HERM ? 8 : 4) : (WA * TC <= 4 ? 2 : 1);
    constexpr int CW = 16 * TC, RS = 4 * NSUB;   // columns of the macro tile; rows of the workgroup's step
    extern __shared__ double2 gsm[];             // 16 TA x 16 TC, then the borders: 16 TA, 16 TC, 1
    const int lane = threadIdx.x & 63, wv = wave_id();
    const int h = wv % GA, sub = wv / GA;
    const int64_t b = blockIdx.z;
    const int mt = tile0 + (int)blockIdx.y, a0 = (mt / ntc) * (16 * TA), c0 = (mt % ntc) * CW;
    const int aw = a0 + 16 * WA * h;             // first row of G of this wave
    const int64_t r_begin = (int64_t)blockIdx.x * chunk;
    const int64_t r_end = r_begin + chunk < nrows ? r_begin + chunk : nrows;
    const int kr = lane >> 4, cl = lane & 15;
    // the macro tiles of the last row and column of tiles carry the border
    const bool do_a = BORD && !HERM && a0 + 16 * TA >= na - 1, do_c = BORD && c0 + CW >= nc - 1;
    const int na_t = BORD ? na - 1 : na, nc_t = BORD ? nc - 1 : nc;
    bool aok[WA], cok[TC];
    int ao[WA], co[TC];                          // column offsets, clamped
#pragma unroll
    for (int t = 0; t < WA; ++t) {
        aok[t] = aw + 16 * t + cl < na_t;
        ao[t] = aok[t] ? aw + 16 * t + cl : na_t - 1;
    }
#pragma unroll
    for (int u = 0; u < TC; ++u) {
        cok[u] = c0 + 16 * u + cl < nc_t;
        co[u] = cok[u] ? c0 + 16 * u + cl : nc_t - 1;
    }
    dvec4 gr[WA][TC], gi[WA][TC];
#pragma unroll
    for (int t = 0; t < WA; ++t)
#pragma unroll
        for (int u = 0; u < TC; ++u) { gr[t][u] = (dvec4){0, 0, 0, 0}; gi[t][u] = (dvec4){0, 0, 0, 0}; }
    double2 ba[WA], bc[TC], bb = make_double2(0, 0);   // border column G(a, nc-1), border row G(na-1, c), corner
#pragma unroll
    for (int t = 0; t < WA; ++t) ba[t] = make_double2(0, 0);
#pragma unroll
    for (int u = 0; u < TC; ++u) bc[u] = make_double2(0, 0);
    double2 xv[PF][WA], zv[PF][TC], xe[PF], ze[PF];
    bool okv[PF];
    const double2 *Xb = X + b * xb, *Zb = Z + b * zb;
    auto load = [&](int p, int64_t r0) {
        int64_t r = r0 + kr;
        okv[p] = r < r_end;
        if (!okv[p]) r = r_end - 1;
        const double2 *xp = Xb + r * xr;
#pragma unroll
        for (int t = 0; t < WA; ++t) {
            if constexpr (TA * TC == 1 && HERM) {
                const dvec2 v = __builtin_nontemporal_load((const dvec2 *)(xp + ao[t]));
                xv[p][t] = make_double2(v.x, v.y);
            } else xv[p][t] = xp[ao[t]];
        }
        if constexpr (!HERM) {
            const double2 *zp = Zb + r * zr;
#pragma unroll
            for (int u = 0; u < TC; ++u) zv[p][u] = zp[co[u]];
            if constexpr (BORD) { ze[p] = zp[nc - 1]; xe[p] = xp[na - 1]; }
        } else if constexpr (BORD) {
            ze[p] = xp[na - 1];
        }
    };
    const int64_t rw = r_begin + 4 * sub;
#pragma unroll
    for (int p = 0; p < PF; ++p) load(p, rw + RS * p);
    for (int64_t r0 = rw; r0 < r_end; r0 += RS * PF) {
#pragma unroll
        for (int p = 0; p < PF; ++p) {
            double2 x[WA], z[TC], xb1 = make_double2(0, 0), zb1 = make_double2(0, 0);
#pragma unroll
            for (int t = 0; t < WA; ++t) {
                const bool ok = okv[p] && aok[t];
                x[t] = make_double2(ok ? xv[p][t].x : 0.0, ok ? xv[p][t].y : 0.0);
            }
#pragma unroll
            for (int u = 0; u < TC; ++u) {
                if constexpr (HERM) z[u] = x[u];
                else {
                    const bool ok = okv[p] && cok[u];
                    z[u] = make_double2(ok ? zv[p][u].x : 0.0, ok ? zv[p][u].y : 0.0);
                }
            }
            if constexpr (BORD) {
                zb1 = make_double2(okv[p] ? ze[p].x : 0.0, okv[p] ? ze[p].y : 0.0);
                if constexpr (HERM) xb1 = zb1;
                else xb1 = make_double2(okv[p] ? xe[p].x : 0.0, okv[p] ? xe[p].y : 0.0);
            }
            load(p, r0 + RS * (p + PF));         // rows past the chunk count as zeros
#pragma unroll
            for (int t = 0; t < WA; ++t)
#pragma unroll
                for (int u = HERM ? t : 0; u < TC; ++u) {
                    gr[t][u] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[t].x, z[u].x, gr[t][u], 0, 0, 0);
                    gi[t][u] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[t].x, z[u].y, gi[t][u], 0, 0, 0);
                }
#pragma unroll
            for (int t = 0; t < WA; ++t)
#pragma unroll
                for (int u = HERM ? t : 0; u < TC; ++u) {
                    gr[t][u] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[t].y, z[u].y, gr[t][u], 0, 0, 0);
                    gi[t][u] = __builtin_amdgcn_mfma_f64_16x16x4f64(-x[t].y, z[u].x, gi[t][u], 0, 0, 0);
                }
            if constexpr (BORD) {
                if (do_c) {
#pragma unroll
                    for (int t = 0; t < WA; ++t) ba[t] = zadd(ba[t], zcmul(x[t], zb1));
                }
                if (do_a && h == 0) {
#pragma unroll
                    for (int u = 0; u < TC; ++u) bc[u] = zadd(bc[u], zcmul(xb1, z[u]));
                }
                bb = zadd(bb, zcmul(xb1, zb1));
            }
        }
    }
    // the waves' sums, in a fixed order
    double2 *sba = gsm + 16 * TA * CW, *sbc = sba + 16 * TA;
    if constexpr (BORD) {                         // sum the four row classes of a step
        auto rsum = [](double2 v) {
            v.x += __shfl_xor(v.x, 16, 64); v.y += __shfl_xor(v.y, 16, 64);
            v.x += __shfl_xor(v.x, 32, 64); v.y += __shfl_xor(v.y, 32, 64);
            return v;
        };
#pragma unroll
        for (int t = 0; t < WA; ++t) ba[t] = rsum(ba[t]);
#pragma unroll
        for (int u = 0; u < TC; ++u) bc[u] = rsum(bc[u]);
        bb = rsum(bb);
    }
#pragma unroll 1
    for (int w = 0; w < NSUB; ++w) {
        if (sub == w) {
#pragma unroll
            for (int t = 0; t < WA; ++t) {
#pragma unroll
                for (int u = HERM ? t : 0; u < TC; ++u)
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        double2 *o = gsm + (16 * (WA * h + t) + 4 * j + kr) * CW + 16 * u + cl;
                        double2 v = make_double2(gr[t][u][j], gi[t][u][j]);
                        if (w) v = zadd(*o, v);
                        *o = v;
                    }
                __builtin_amdgcn_sched_barrier(0);      // one tile row's sums in registers at a time
            }
            if constexpr (BORD) {
                if (kr == 0) {
#pragma unroll
                    for (int t = 0; t < WA; ++t) {
                        double2 *o = sba + 16 * (WA * h + t) + cl;
                        *o = w ? zadd(*o, ba[t]) : ba[t];
                    }
                    if (h == 0) {
#pragma unroll
                        for (int u = 0; u < TC; ++u) sbc[16 * u + cl] = w ? zadd(sbc[16 * u + cl], bc[u]) : bc[u];
                        if (cl == 0) sbc[CW] = w ? zadd(sbc[CW], bb) : bb;
                    }
                }
            }
        }
        __syncthreads();
    }
    double2 *pb = part + (b * gridDim.x + blockIdx.x) * (int64_t)na * nc;
    for (int e = threadIdx.x; e < 16 * TA * CW; e += 256) {
        const int a = e / CW, c = e % CW;
        if (HERM && a / 16 > c / 16) continue;
        if (a0 + a < na_t && c0 + c < nc_t) pb[(int64_t)(a0 + a) * nc + c0 + c] = gsm[e];
    }
    if constexpr (BORD) {
        const int e = threadIdx.x;
        if (do_c && e < 16 * TA && a0 + e < na_t) pb[(int64_t)(a0 + e) * nc + nc - 1] = sba[e];
        if (do_a && e < CW && c0 + e < nc_t) pb[(int64_t)(na - 1) * nc + c0 + e] = sbc[e];
        if (do_c && (do_a || HERM) && e == 0) pb[(int64_t)(na - 1) * nc + nc - 1] = sbc[CW];
    }
}

static dim3 bgram_reduce_grid(int64_t entries, int64_t nbatch)
{
    const int64_t gx = (entries + 31) / 32;
    return dim3((unsigned)(gx < (1 << 20) ? gx : 1 << 20), (unsigned)nbatch);
}

// Partials that rsvdt_hip_bgram_work_bytes has room for (the plans below use
// at most as many): about 2048 workgroups of four tiles of up to 48 x 48.
static int64_t bgram_work_parts(int64_t nbatch, int64_t nrows, int64_t na, int64_t nc)
{
    auto side = [](int64_t n) { return n <= 16 ? 16 : (n <= 32 ? 32 : 48); };
    const int64_t ntiles = ((na + side(na) - 1) / side(na)) * ((nc + side(nc) - 1) / side(nc));
    const int64_t nsub = ntiles >= 4 ? 1 : (ntiles >= 2 ? 2 : 4);
    const int64_t wg_per_chunk = ((ntiles + (4 / nsub) - 1) / (4 / nsub)) * nbatch;
    const int64_t nch = (2048 + wg_per_chunk - 1) / wg_per_chunk;
    int64_t chunk = (nrows + nch - 1) / nch;
    if (chunk < 64) chunk = 64;
    chunk = (chunk + 3) / 4 * 4;
    return (nrows + chunk - 1) / chunk * nsub;
}

struct bgram_mfma_plan {
    int TA, TC, ntc, ntiles, bord, herm;
    int64_t chunk, nch;
};

// Macro tiles of at most 4 x 4 MFMA tiles, as even as the tile counts allow;
// row chunks so that the grid holds two workgroups per SIMD's worth of waves
// for the large tiles (one fits at a time) and eight per CU for a single tile,
// which needs the loads of many waves in flight.
static bgram_mfma_plan bgram_mfma_shape(int64_t nbatch, int64_t nrows, int64_t na, int64_t nc, bool herm)
{
    bgram_mfma_plan p;
    p.bord = na > 16 && nc > 16 && na % 16 == 1 && nc % 16 == 1;
    const int ta = (int)(p.bord ? na / 16 : (na + 15) / 16), tc = (int)(p.bord ? nc / 16 : (nc + 15) / 16);
    const int ma = (ta + 3) / 4, mc = (tc + 3) / 4;
    p.TA = (ta + ma - 1) / ma;
    p.TC = (tc + mc - 1) / mc;
    p.ntc = mc;
    p.ntiles = ma * mc;
    p.herm = herm && p.ntiles == 1;
    const int64_t target = p.TA * p.TC <= 4 ? 1024 : 512;
    int64_t nch = (target + p.ntiles * nbatch - 1) / (p.ntiles * nbatch);
    const int64_t room = bgram_work_parts(nbatch, nrows, na, nc);
    if (nch > room) nch = room;
    int64_t chunk = (nrows + nch - 1) / nch;
    if (chunk < 64) chunk = 64;
    chunk = (chunk + 15) / 16 * 16;
    p.chunk = chunk;
    p.nch = (nrows + chunk - 1) / chunk;
    return p;
}

template <int TA, int TC, bool HERM, bool BORD>
static int launch_bgram_mfma(const bgram_mfma_plan &p, int64_t nbatch, int64_t nrows, int64_t na, int64_t nc,
                             const double2 *X, int64_t xb, int64_t xr, const double2 *Z, int64_t zb, int64_t zr,
                             double2 *part, hipStream_t s)
{
    const size_t lds = (size_t)(256 * TA * TC + 16 * TA + 16 * TC + 1) * 16;
    for (int t0 = 0; t0 < p.ntiles; t0 += 65535) {     // what a launch takes in this dimension
        const unsigned gy = (unsigned)(p.ntiles - t0 < 65535 ? p.ntiles - t0 : 65535);
        hipLaunchKernelGGL((k_bgram_mfma<TA, TC, HERM, BORD>), dim3((unsigned)p.nch, gy, (unsigned)nbatch), dim3(256), lds,
                           s, nrows, (int)na, (int)nc, p.chunk, t0, p.ntc, X, xb, xr, Z, zb, zr, part);
    }
    RSVDT_LAUNCH_CHECK("rsvdt_hip_bgram(mfma)");
    return RSVDT_HIP_OK;
}

static int64_t bgram_chunk(int64_t nbatch, int64_t nrows, int64_t na, int64_t nc)
{
    // aim for ~2048 workgroups in flight in total, chunks of >= 256 rows
    const int64_t tiles = ((na + BG_T - 1) / BG_T) * ((nc + BG_T - 1) / BG_T) * nbatch;
    int64_t nch = (4096 + tiles - 1) / tiles;
    if (nch < 1) nch = 1;
    int64_t chunk = (nrows + nch - 1) / nch;
    if (chunk < 256) chunk = 256;
    chunk = (chunk + BG_T - 1) / BG_T * BG_T;
    return chunk;
}

// ----------------------------------------------------------------- bapply
__global__ __launch_bounds__(256) void k_bapply(
    int64_t nrows, int64_t na, int64_t nc, int ncpad, int rb,
    const double2 *X, int64_t xb, int64_t xr, int64_t xa, const double2 *__restrict__ C, double alpha,
    const double2 *Y, int64_t yb, int64_t yr, int64_t yc, double2 *Out, int64_t ob, int64_t orow, int64_t oc)
{
    extern __shared__ double2 sxr[];          // rb x na
    const int64_t b = blockIdx.y;
    const int64_t r0 = (int64_t)blockIdx.x * rb;
    const double2 *Xb = X + b * xb;
    for (int i = threadIdx.x; i < rb * na; i += blockDim.x) {
        const int rr = i / (int)na, a = i % (int)na;
        const int64_t r = r0 + rr;
        sxr[i] = (r < nrows) ? Xb[r * xr + a * xa] : make_double2(0, 0);
    }
    __syncthreads();
    const int rr = threadIdx.x / ncpad, c = threadIdx.x % ncpad;
    const int64_t r = r0 + rr;
    if (rr >= rb || r >= nrows || c >= nc) return;
    const double2 *Cb = C + b * na * nc;
    double2 acc = make_double2(0, 0);
    if (Y != nullptr) {
        const double2 yv = Y[b * yb + r * yr + c * yc];
        acc.x = alpha * yv.x; acc.y = alpha * yv.y;
    }
    const double2 *xrow = sxr + rr * na;
    for (int64_t a = 0; a < na; ++a) {
        const double2 xv = xrow[a], cv = Cb[a * nc + c];
        acc.x += xv.x * cv.x - xv.y * cv.y;
        acc.y += xv.x * cv.y + xv.y * cv.x;
    }
    Out[b * ob + r * orow + c * oc] = acc;
}

// FP64 MFMA batched apply for unit column strides:
//   Out_b(r, c) = alpha Y_b(r, c) + sum_a X_b(r, a) C_b(a, c).
// grid.y = column tile of 16 TC columns; the workgroup stages C_b(:, tile) in
// LDS once and its waves walk 16-row tiles (grid-stride).  A(16x4): lane i ->
// X(r0 + i%16, a0 + i/16); B(4x16): lane i -> C(a0 + i/16, c0 + i%16);
// D: lane i holds Out(r0 + 4j + i/16, c0 + i%16).  The (row tile, 4-column
// step) sequence of a wave is one stream with PF steps of X in flight, across
// tile boundaries too.  With one column tile a wave's loads of a row tile are
// all issued before it writes the tile, and no other wave reads those rows, so
// Out may alias X; Out may always alias Y (read and written by the same lane).
// BORD: a last column beyond the 16-wide tiles (nc = 16 T + 1, the bases of
// Nw + 1 snapshots) is a plain FMA sum on the operands the lanes hold.
// Bound by memory and FP64 MFMA together at 32 columns (MFMAs busy in 51 to 55 % of
// the cycles, 45 to 47 % with Y), by MFMA above.  8 batches of 98,304 x 65 times 65 x 32:
// alone 340 us, with Y 372 us (413 and 520 us with one step in flight); in a
// projection, after other kernels, 366 and 411 us, 3.3 and 3.9 TB/s.  PF = 8 is
// slower (385 us), 16 x 16 chunks turned through LDS too (383 us).
template <int TC, bool BORD>
__global__ __launch_bounds__(256) void k_bapply_mfma(
    int64_t nrows, int na, int nc, const double2 *X, int64_t xb, int64_t xr,
    const double2 *__restrict__ C, double alpha, const double2 *Y, int64_t yb, int64_t yr,
    double2 *Out, int64_t ob, int64_t orow)
{
    extern __shared__ double2 cs_b[];               // [na4][16 TC], then the border column [na4]
    constexpr int CW = 16 * TC, PF = 4;
    const int lane = threadIdx.x & 63, wv = wave_id();
    const int64_t b = blockIdx.z;
    const int c0 = (int)blockIdx.y * CW;
    const int na4 = (na + 3) & ~3, nks = na4 >> 2;
    const int nc_t = BORD ? nc - 1 : nc;            // columns in tiles
    const bool do_b = BORD && blockIdx.y == gridDim.y - 1;
    const double2 *Cb = C + b * na * nc;
    for (int e = threadIdx.x; e < na4 * CW; e += 256) {
        const int a = e / CW, c = c0 + e % CW;
        double2 v = make_double2(0, 0);
        if (a < na && c < nc_t) v = Cb[(int64_t)a * nc + c];
        cs_b[e] = v;
    }
    double2 *cb_l = cs_b + (int64_t)na4 * CW;
    if constexpr (BORD) {
        for (int a = threadIdx.x; a < na4; a += 256) {
            double2 v = make_double2(0, 0);
            if (a < na) v = Cb[(int64_t)a * nc + nc - 1];
            cb_l[a] = v;
        }
    }
    __syncthreads();
    const int kr = lane >> 4, cl = lane & 15;
    const double2 *Xb = X + b * xb;
    const int64_t ntile = (nrows + 15) / 16, step = (int64_t)gridDim.x * 4;
    int64_t tile = (int64_t)blockIdx.x * 4 + wv;
    if (tile >= ntile) return;
    // load position: step ls of row tile lt (clamped to the last tile and row)
    int64_t lt = tile;
    int ls = 0;
    auto row_ptr = [&](int64_t t) {
        int64_t r = (t < ntile ? t : ntile - 1) * 16 + cl;
        if (r >= nrows) r = nrows - 1;
        return Xb + r * xr;
    };
    const double2 *lp = row_ptr(lt);
    double2 ring[PF];
    auto load = [&](int p) {
        const int a = 4 * ls + kr;
        ring[p] = lp[a < na ? a : na - 1];
        if (++ls == nks) { ls = 0; lt += step; lp = row_ptr(lt); }
    };
#pragma unroll
    for (int p = 0; p < PF; ++p) load(p);
    dvec4 dr[TC], di[TC];
    double2 bd = make_double2(0, 0);
#pragma unroll
    for (int u = 0; u < TC; ++u) { dr[u] = (dvec4){0, 0, 0, 0}; di[u] = (dvec4){0, 0, 0, 0}; }
    int ks = 0;
    while (tile < ntile) {
#pragma unroll
        for (int p = 0; p < PF; ++p) {
            if (tile < ntile) {
                const int a = 4 * ks + kr;
                const bool ok = a < na;             // a column past the end has no product (X may hold anything there)
                const double2 x = make_double2(ok ? ring[p].x : 0.0, ok ? ring[p].y : 0.0);
                load(p);
                const double2 *crow = cs_b + a * CW + cl;
                double2 cv[TC];
#pragma unroll
                for (int u = 0; u < TC; ++u) cv[u] = crow[16 * u];
#pragma unroll
                for (int u = 0; u < TC; ++u) {
                    dr[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.x, cv[u].x, dr[u], 0, 0, 0);
                    di[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.x, cv[u].y, di[u], 0, 0, 0);
                }
#pragma unroll
                for (int u = 0; u < TC; ++u) {
                    dr[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(-x.y, cv[u].y, dr[u], 0, 0, 0);
                    di[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.y, cv[u].x, di[u], 0, 0, 0);
                }
                if constexpr (BORD) {
                    if (do_b) bd = zadd(bd, zmul(x, cb_l[a]));
                }
                if (++ks == nks) {                  // tile done: store and restart the sums
                    const int64_t r0 = tile * 16;
                    double2 yv[4][TC];              // clamped addresses: all loads in flight at once
                    if (Y != nullptr) {
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            const int64_t r = r0 + 4 * j + kr < nrows ? r0 + 4 * j + kr : nrows - 1;
#pragma unroll
                            for (int u = 0; u < TC; ++u) {
                                const int c = c0 + 16 * u + cl < nc_t ? c0 + 16 * u + cl : nc_t - 1;
                                yv[j][u] = Y[b * yb + r * yr + c];
                            }
                        }
                    } else {
#pragma unroll
                        for (int j = 0; j < 4; ++j)
#pragma unroll
                            for (int u = 0; u < TC; ++u) yv[j][u] = make_double2(0, 0);
                    }
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const int64_t r = r0 + 4 * j + kr;
#pragma unroll
                        for (int u = 0; u < TC; ++u) {
                            const int c = c0 + 16 * u + cl;
                            double2 o = make_double2(dr[u][j], di[u][j]);
                            if (Y != nullptr) { o.x += alpha * yv[j][u].x; o.y += alpha * yv[j][u].y; }
                            if (r < nrows && c < nc_t) Out[b * ob + r * orow + c] = o;
                        }
                    }
                    if constexpr (BORD) {
                        if (do_b) {
                            bd.x += __shfl_xor(bd.x, 16, 64); bd.y += __shfl_xor(bd.y, 16, 64);
                            bd.x += __shfl_xor(bd.x, 32, 64); bd.y += __shfl_xor(bd.y, 32, 64);
                            const int64_t r = r0 + cl;
                            if (kr == 0 && r < nrows) {
                                if (Y != nullptr) {
                                    const double2 yv = Y[b * yb + r * yr + nc - 1];
                                    bd.x += alpha * yv.x; bd.y += alpha * yv.y;
                                }
                                Out[b * ob + r * orow + nc - 1] = bd;
                            }
                            bd = make_double2(0, 0);
                        }
                    }
                    ks = 0;
                    tile += step;
#pragma unroll
                    for (int u = 0; u < TC; ++u) { dr[u] = (dvec4){0, 0, 0, 0}; di[u] = (dvec4){0, 0, 0, 0}; }
                }
            }
        }
    }
}

// One CholeskyQR step on the rows: Out_b = X_b C_b with C_b upper triangular
// (n <= 16 TC <= 64), and with GRAM the Gram matrix of the result,
// Out_b^H Out_b, from the same registers: lane i of the apply's accumulators
// holds Out(r0 + 4j + i/16, c0 + i%16), which is exactly the operand layout of
// the Gram's 4-row step j, so the next pass's Gram costs MFMAs but no memory.
// A wave walks 16 RT-row tiles, the next tile's rows loaded while the current
// one computes; it reads all of a tile before it writes any of it and no other
// wave touches its rows, so Out may be X.  The zero tiles of C are skipped.
// The waves' Gram sums meet in LDS in wave order and go to k_bgram_reduce as
// one partial per workgroup.  NT: nontemporal loads and stores for blocks
// beyond the last-level cache.  Without GRAM (the last pass) the apply alone.
// Bound by memory for 16 columns, by FP64 MFMA above.  16 blocks of
// 393,216 x 16: 622 us, 5.2 TB/s (apply 612 us, then the Gram 329 us, as two
// kernels); a whole QR of 32 blocks of 60,000 x 32 went from 3642 to 1984 us.
template <int TC, bool GRAM, bool NT>
__global__ __launch_bounds__(256) void k_bapply_gram(int64_t nrows, int n, const double2 *X, int64_t xb, int64_t xr,
                                                     const double2 *__restrict__ C, double2 *Out,
                                                     double2 *__restrict__ part)
{
    constexpr int RT = TC == 1 ? 2 : 1, CW = 16 * TC, NS = 4 * TC;
    extern __shared__ double2 gsm[];             // C_b [CW][CW], then the workgroup's Gram sums
    const int lane = threadIdx.x & 63, wv = wave_id(), kr = lane >> 4, cl = lane & 15;
    const int64_t b = blockIdx.z;
    const double2 *Cb = C + b * n * n;
    for (int e = threadIdx.x; e < CW * CW; e += 256) {
        const int a = e / CW, c = e % CW;
        double2 v = make_double2(0, 0);
        if (a < n && c < n) v = Cb[a * n + c];
        gsm[e] = v;
    }
    __syncthreads();
    const double2 *Xb = X + b * xb;
    double2 *Ob = Out + b * xb;
    int ao[NS];
    bool aok[NS];
#pragma unroll
    for (int q = 0; q < NS; ++q) {
        aok[q] = 4 * q + kr < n;
        ao[q] = aok[q] ? 4 * q + kr : n - 1;
    }
    double2 xn[RT][NS];
    bool rn[RT];
    auto load = [&](int64_t tile) {
#pragma unroll
        for (int t = 0; t < RT; ++t) {
            int64_t r = tile * (16 * RT) + 16 * t + cl;
            rn[t] = r < nrows;
            if (!rn[t]) r = nrows - 1;
            const double2 *xp = Xb + r * xr;
#pragma unroll
            for (int q = 0; q < NS; ++q) {
                if constexpr (NT) {
                    const dvec2 v = __builtin_nontemporal_load((const dvec2 *)(xp + ao[q]));
                    xn[t][q] = make_double2(v.x, v.y);
                } else xn[t][q] = xp[ao[q]];
            }
        }
    };
    dvec4 gr[TC][TC], gi[TC][TC];
#pragma unroll
    for (int t = 0; t < TC; ++t)
#pragma unroll
        for (int u = 0; u < TC; ++u) { gr[t][u] = (dvec4){0, 0, 0, 0}; gi[t][u] = (dvec4){0, 0, 0, 0}; }
    const int64_t ntile = (nrows + 16 * RT - 1) / (16 * RT), step = (int64_t)gridDim.x * 4;
    int64_t tile = (int64_t)blockIdx.x * 4 + wv;
    if (tile < ntile) load(tile);
    for (; tile < ntile; tile += step) {
        double2 x[RT][NS];
#pragma unroll
        for (int t = 0; t < RT; ++t)
#pragma unroll
            for (int q = 0; q < NS; ++q) {
                const bool ok = rn[t] && aok[q];
                x[t][q] = make_double2(ok ? xn[t][q].x : 0.0, ok ? xn[t][q].y : 0.0);
            }
        load(tile + step < ntile ? tile + step : tile);       // the last one again: its values are not used
        dvec4 dr[RT][TC], di[RT][TC];
#pragma unroll
        for (int t = 0; t < RT; ++t)
#pragma unroll
            for (int u = 0; u < TC; ++u) { dr[t][u] = (dvec4){0, 0, 0, 0}; di[t][u] = (dvec4){0, 0, 0, 0}; }
#pragma unroll
        for (int q = 0; q < NS; ++q)
#pragma unroll
            for (int u = q / 4; u < TC; ++u) {   // C(a, c) = 0 for a > c
                const double2 cv = gsm[(4 * q + kr) * CW + 16 * u + cl];
#pragma unroll
                for (int t = 0; t < RT; ++t) {
                    dr[t][u] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[t][q].x, cv.x, dr[t][u], 0, 0, 0);
                    di[t][u] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[t][q].x, cv.y, di[t][u], 0, 0, 0);
                }
#pragma unroll
                for (int t = 0; t < RT; ++t) {
                    dr[t][u] = __builtin_amdgcn_mfma_f64_16x16x4f64(-x[t][q].y, cv.y, dr[t][u], 0, 0, 0);
                    di[t][u] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[t][q].y, cv.x, di[t][u], 0, 0, 0);
                }
            }
        const int64_t r0 = tile * (16 * RT);
#pragma unroll
        for (int t = 0; t < RT; ++t)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int64_t r = r0 + 16 * t + 4 * j + kr;
                if (r < nrows) {
#pragma unroll
                    for (int u = 0; u < TC; ++u)
                        if (16 * u + cl < n) {
                            double2 *o = Ob + r * xr + 16 * u + cl;
                            if constexpr (NT) {
                                const dvec2 v = {dr[t][u][j], di[t][u][j]};
                                __builtin_nontemporal_store(v, (dvec2 *)o);
                            } else *o = make_double2(dr[t][u][j], di[t][u][j]);
                        }
                }
            }
        if constexpr (GRAM) {
#pragma unroll
            for (int t = 0; t < RT; ++t)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
#pragma unroll
                    for (int u = 0; u < TC; ++u)
#pragma unroll
                        for (int v = u; v < TC; ++v) {
                            gr[u][v] = __builtin_amdgcn_mfma_f64_16x16x4f64(dr[t][u][j], dr[t][v][j], gr[u][v], 0, 0, 0);
                            gi[u][v] = __builtin_amdgcn_mfma_f64_16x16x4f64(dr[t][u][j], di[t][v][j], gi[u][v], 0, 0, 0);
                        }
#pragma unroll
                    for (int u = 0; u < TC; ++u)
#pragma unroll
                        for (int v = u; v < TC; ++v) {
                            gr[u][v] = __builtin_amdgcn_mfma_f64_16x16x4f64(di[t][u][j], di[t][v][j], gr[u][v], 0, 0, 0);
                            gi[u][v] = __builtin_amdgcn_mfma_f64_16x16x4f64(-di[t][u][j], dr[t][v][j], gi[u][v], 0, 0, 0);
                        }
                }
        }
    }
    if constexpr (GRAM) {
        __syncthreads();                          // C_b is no longer read
#pragma unroll 1
        for (int w = 0; w < 4; ++w) {
            if (wv == w) {
#pragma unroll
                for (int u = 0; u < TC; ++u) {
#pragma unroll
                    for (int v = u; v < TC; ++v)
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            double2 *o = gsm + (16 * u + 4 * j + kr) * CW + 16 * v + cl;
                            double2 g = make_double2(gr[u][v][j], gi[u][v][j]);
                            if (w) g = zadd(*o, g);
                            *o = g;
                        }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            __syncthreads();
        }
        double2 *pb = part + (b * gridDim.x + blockIdx.x) * (int64_t)n * n;
        for (int e = threadIdx.x; e < CW * CW; e += 256) {
            const int a = e / CW, c = e % CW;
            if (a / 16 <= c / 16 && a < n && c < n) pb[a * n + c] = gsm[e];
        }
    }
}

// Dense propagator times N x k blocks: Out_b = E X_b (+ F_b), E an N x N
// row-major matrix, the blocks' columns taken together as nb*k columns.  A
// workgroup owns ROWS rows and 16 CT columns; its 8 waves take every eighth
// 4-column step of E (the product is a few MFLOP and follows the previous one
// on the stream, so the reduction is split for latency, not for work) and
// their sums meet in LDS in wave order.  PF steps of both operands are in
// flight per wave.  With one column tile the FP64 MFMAs of 16 rows would take 3.4
// us on the few CUs that have work: ROWS = 4 spreads them over four times as many
// with the 4x4x4 MFMA, its four blocks the tile's four groups of columns (lane i
// holds A[i%4][i/16], B[i/16][i%16], D[i/16][i%16]; checked with known products).
// N = 500, k = 10: 6.6 us (7.8 with 16 rows); 650 columns (CT = 2): 35 us.
template <int CT, int ROWS>
__global__ __launch_bounds__(512) void k_dense_apply(int N, int k, int ncol, const double2 *__restrict__ E,
                                                     const double2 *__restrict__ X, const double2 *__restrict__ F,
                                                     double2 *__restrict__ Out)
{
    using acc = typename std::conditional<ROWS == 16, dvec4, double>::type;
    constexpr int PF = CT == 1 ? 8 : 4, CW = 16 * CT;
    __shared__ double2 red[8][ROWS][CW];
    const int lane = threadIdx.x & 63, wv = wave_id(), kr = lane >> 4, cl = lane & 15;
    const int r0 = blockIdx.x * ROWS, c0 = blockIdx.y * CW;
    const int64_t bs = (int64_t)N * k;
    const double2 *er = E + (int64_t)min(r0 + cl % ROWS, N - 1) * N;
    const double2 *xc[CT];
#pragma unroll
    for (int u = 0; u < CT; ++u) {
        const int c = min(c0 + 16 * u + cl, ncol - 1);      // columns past the end repeat the last, never stored
        xc[u] = X + (int64_t)(c / k) * bs + c % k;
    }
    double2 ev[PF], xv[PF][CT];
    auto load = [&](int p, int q) {
        const int a = min(q + kr, N - 1);
        ev[p] = er[a];
#pragma unroll
        for (int u = 0; u < CT; ++u) xv[p][u] = xc[u][(int64_t)a * k];
    };
    auto mfma = [](double x, double y, acc c) -> acc {
        if constexpr (ROWS == 16) return __builtin_amdgcn_mfma_f64_16x16x4f64(x, y, c, 0, 0, 0);
        else return __builtin_amdgcn_mfma_f64_4x4x4f64(x, y, c, 0, 0, 0);
    };
    acc dr[CT], di[CT];
#pragma unroll
    for (int u = 0; u < CT; ++u) { dr[u] = acc{}; di[u] = acc{}; }
#pragma unroll
    for (int p = 0; p < PF; ++p) load(p, 4 * wv + 32 * p);
    for (int q0 = 4 * wv; q0 < N; q0 += 32 * PF) {
#pragma unroll
        for (int p = 0; p < PF; ++p) {
            const int q = q0 + 32 * p;
            const bool ok = q + kr < N;          // steps past the end multiply zeros
            const double2 e = make_double2(ok ? ev[p].x : 0.0, ok ? ev[p].y : 0.0);
            double2 x[CT];
#pragma unroll
            for (int u = 0; u < CT; ++u) x[u] = make_double2(ok ? xv[p][u].x : 0.0, ok ? xv[p][u].y : 0.0);
            load(p, q + 32 * PF);
#pragma unroll
            for (int u = 0; u < CT; ++u) {
                dr[u] = mfma(e.x, x[u].x, dr[u]);
                di[u] = mfma(e.x, x[u].y, di[u]);
            }
#pragma unroll
            for (int u = 0; u < CT; ++u) {
                dr[u] = mfma(-e.y, x[u].y, dr[u]);
                di[u] = mfma(e.y, x[u].x, di[u]);
            }
        }
    }
#pragma unroll
    for (int u = 0; u < CT; ++u) {
        if constexpr (ROWS == 16) {
#pragma unroll
            for (int j = 0; j < 4; ++j) red[wv][4 * j + kr][16 * u + cl] = make_double2(dr[u][j], di[u][j]);
        } else red[wv][kr][16 * u + cl] = make_double2(dr[u], di[u]);
    }
    __syncthreads();
    for (int e = threadIdx.x; e < ROWS * CW; e += 512) {
        const int r = r0 + e / CW, c = c0 + e % CW;
        if (r >= N || c >= ncol) continue;
        double2 s = red[0][e / CW][e % CW];
#pragma unroll
        for (int w = 1; w < 8; ++w) s = zadd(s, red[w][e / CW][e % CW]);
        const int64_t idx = (int64_t)(c / k) * bs + (int64_t)r * k + c % k;
        if (F != nullptr) s = zadd(s, F[idx]);
        Out[idx] = s;
    }
}

}  // namespace rsvdt

using namespace rsvdt;

extern "C" int rsvdt_hip_coef_gemm(int64_t P, int64_t K, int64_t L, const double *coef, int64_t cq, int64_t cp,
                                   int64_t p0, int sgn, int64_t cmod, double alpha, const double *in, int64_t ldi,
                                   void *out, int64_t ldo, int out_prec, double beta, rsvdt_stream_t s)
{
    if (P <= 0 || L <= 0) return RSVDT_HIP_OK;
    if (K <= 0 || cmod <= 0 || (out_prec != 64 && out_prec != 32) || P > 65535LL * 16) {
        set_error_msg("rsvdt_hip_coef_gemm: bad arguments");
        return RSVDT_HIP_ERR_ARG;
    }
    hipStream_t st = as_stream(s);
    const int64_t Kpad = (K + 3) & ~(int64_t)3;
    // LDS of the coefficient block for a row tile of 16 T rows (padded pitch)
    auto lds_of = [Kpad](int T) { return Kpad * (16 * T + 4) * 16; };
    if (lds_of(1) > 150 * 1024) {
        set_error_msg("rsvdt_hip_coef_gemm: K too large for the LDS coefficient block (K <= 480)");
        return RSVDT_HIP_ERR_ARG;
    }
    // widest row tile whose coefficient block fits in 144 KB of LDS
    if (P > 64 && lds_of(8) <= 144 * 1024)
        return launch_coef<8>(P, K, L, coef, cq, cp, p0, sgn, cmod, alpha, in, ldi, out, ldo, out_prec, beta, st);
    if (P > 32 && lds_of(4) <= 144 * 1024)
        return launch_coef<4>(P, K, L, coef, cq, cp, p0, sgn, cmod, alpha, in, ldi, out, ldo, out_prec, beta, st);
    if (P > 16 && lds_of(2) <= 144 * 1024)
        return launch_coef<2>(P, K, L, coef, cq, cp, p0, sgn, cmod, alpha, in, ldi, out, ldo, out_prec, beta, st);
    return launch_coef<1>(P, K, L, coef, cq, cp, p0, sgn, cmod, alpha, in, ldi, out, ldo, out_prec, beta, st);
}

extern "C" size_t rsvdt_hip_bgram_work_bytes(int64_t nbatch, int64_t nrows, int64_t na, int64_t nc)
{
    const int64_t chunk = bgram_chunk(nbatch, nrows, na, nc);
    const int64_t nch = (nrows + chunk - 1) / chunk;
    int64_t parts = bgram_work_parts(nbatch, nrows, na, nc);
    if (nch > parts) parts = nch;
    return (size_t)(nbatch * parts * na * nc) * 16 + 256;
}

extern "C" int rsvdt_hip_bgram(int64_t nbatch, int64_t nrows, int64_t na, int64_t nc, const double *X, int64_t xb,
                               int64_t xr, int64_t xa, const double *Z, int64_t zb, int64_t zr, int64_t zc, double *G,
                               void *work, rsvdt_stream_t s)
{
    if (nbatch <= 0 || na <= 0 || nc <= 0) return RSVDT_HIP_OK;
    if (nrows <= 0) return rsvdt_hip_zero(G, (size_t)(nbatch * na * nc) * 16, s);
    if (nbatch > 65535) { set_error_msg("rsvdt_hip_bgram: nbatch > 65535"); return RSVDT_HIP_ERR_ARG; }
    hipStream_t st = as_stream(s);
    int64_t nparts;
    int herm = 0, ntile = 0;
    if (xa == 1 && zc == 1) {
        const bgram_mfma_plan p =
            bgram_mfma_shape(nbatch, nrows, na, nc, X == Z && na == nc && xr == zr && (xb == zb || nbatch == 1));
        const double2 *X2 = (const double2 *)X, *Z2 = (const double2 *)Z;
        double2 *W = (double2 *)work;
        int rc = RSVDT_HIP_ERR_ARG;
#define RSVDT_BG_L(A, C, H, B) rc = launch_bgram_mfma<A, C, H, B>(p, nbatch, nrows, na, nc, X2, xb, xr, Z2, zb, zr, W, st)
#define RSVDT_BG(A, C)                                                  \
        if (p.TA == A && p.TC == C) {                                   \
            if (p.bord) {                                               \
                if (A == C && p.herm) RSVDT_BG_L(A, C, A == C, true);   \
                else RSVDT_BG_L(A, C, false, true);                     \
            } else {                                                    \
                if (A == C && p.herm) RSVDT_BG_L(A, C, A == C, false);  \
                else RSVDT_BG_L(A, C, false, false);                    \
            }                                                           \
        }
#define RSVDT_BG_ROW(A) RSVDT_BG(A, 1) RSVDT_BG(A, 2) RSVDT_BG(A, 3) RSVDT_BG(A, 4)
        RSVDT_BG_ROW(1) RSVDT_BG_ROW(2) RSVDT_BG_ROW(3) RSVDT_BG_ROW(4)
#undef RSVDT_BG_ROW
#undef RSVDT_BG
#undef RSVDT_BG_L
        if (rc) return rc;
        nparts = p.nch;
        herm = p.herm;
        ntile = p.bord ? (int)(na / 16) : (int)((na + 15) / 16);
    } else {
        const int64_t chunk = bgram_chunk(nbatch, nrows, na, nc);
        const int64_t nch = (nrows + chunk - 1) / chunk;
        const int nta = (int)((na + BG_T - 1) / BG_T), ntc = (int)((nc + BG_T - 1) / BG_T);
        hipLaunchKernelGGL(k_bgram_part, dim3((unsigned)nch, (unsigned)(nta * ntc), (unsigned)nbatch), dim3(256), 0,
                           st, nrows, na, nc, chunk, ntc, (const double2 *)X, xb, xr, xa, (const double2 *)Z, zb, zr,
                           zc, (double2 *)work);
        RSVDT_LAUNCH_CHECK("rsvdt_hip_bgram(part)");
        nparts = nch;
    }
    hipLaunchKernelGGL(k_bgram_reduce, bgram_reduce_grid(na * nc, nbatch), dim3(256), 0, st, nparts, (int)na,
                       (int)nc, herm, ntile, (const double2 *)work, (double2 *)G);
    RSVDT_LAUNCH_CHECK("rsvdt_hip_bgram(reduce)");
    return RSVDT_HIP_OK;
}

template <int TC, bool BORD>
static int launch_bapply_mfma(int64_t nct, int64_t nbatch, int64_t nrows, int64_t na, int64_t nc, const double *X,
                              int64_t xb, int64_t xr, const double *C, double alpha, const double *Y, int64_t yb,
                              int64_t yr, double *Out, int64_t ob, int64_t orow, hipStream_t s)
{
    const int64_t na4 = (na + 3) & ~(int64_t)3;
    const size_t lds = (size_t)na4 * (16 * TC + (BORD ? 1 : 0)) * 16;
    const int64_t ntile = (nrows + 15) / 16;
    int64_t gx = (ntile + 3) / 4;
    const int64_t cap = (1024 + nct * nbatch - 1) / (nct * nbatch);       // four workgroups per CU
    if (gx > cap) gx = cap < 1 ? 1 : cap;
    hipLaunchKernelGGL((k_bapply_mfma<TC, BORD>), dim3((unsigned)gx, (unsigned)nct, (unsigned)nbatch), dim3(256), lds, s,
                       nrows, (int)na, (int)nc, (const double2 *)X, xb, xr, (const double2 *)C, alpha,
                       (const double2 *)Y, yb, yr, (double2 *)Out, ob, orow);
    RSVDT_LAUNCH_CHECK("rsvdt_hip_bapply(mfma)");
    return RSVDT_HIP_OK;
}

extern "C" int rsvdt_hip_bapply(int64_t nbatch, int64_t nrows, int64_t na, int64_t nc, const double *X, int64_t xb,
                                int64_t xr, int64_t xa, const double *C, double alpha, const double *Y, int64_t yb,
                                int64_t yr, int64_t yc, double *Out, int64_t ob, int64_t orow, int64_t oc,
                                rsvdt_stream_t s)
{
    if (nbatch <= 0 || nrows <= 0 || nc <= 0) return RSVDT_HIP_OK;
    if (nbatch > 65535) {
        set_error_msg("rsvdt_hip_bapply: nbatch <= 65535 required");
        return RSVDT_HIP_ERR_ARG;
    }
    hipStream_t st = as_stream(s);
    const bool unit = xa == 1 && oc == 1 && (Y == nullptr || yc == 1);
    const int64_t na4 = (na + 3) & ~(int64_t)3;
    if (unit && na > 0 && na4 * 64 * 16 <= 150 * 1024) {
        // column tiles of at most 64, as even as their number allows; with more
        // than one, rows are read by several workgroups, so not in place (65
        // columns are one tile and a border, and stay refused as before)
        const bool bord = nc > 16 && nc % 16 == 1;
        const int64_t t16 = bord ? nc / 16 : (nc + 15) / 16, nct = (t16 + 3) / 4;
        const int TC = (int)((t16 + nct - 1) / nct);
        if (nc > 64 && X == Out) {
            set_error_msg("rsvdt_hip_bapply: in place needs nc <= 64 with unit strides");
            return RSVDT_HIP_ERR_ARG;
        }
#define RSVDT_BA(T)                                                                                               \
        if (TC == T)                                                                                              \
            return bord ? launch_bapply_mfma<T, true>(nct, nbatch, nrows, na, nc, X, xb, xr, C, alpha, Y, yb, yr, \
                                                      Out, ob, orow, st)                                          \
                        : launch_bapply_mfma<T, false>(nct, nbatch, nrows, na, nc, X, xb, xr, C, alpha, Y, yb,    \
                                                       yr, Out, ob, orow, st);
        RSVDT_BA(1) RSVDT_BA(2) RSVDT_BA(3) RSVDT_BA(4)
#undef RSVDT_BA
    }
    if (nc > 256 || na > 512) {
        set_error_msg("rsvdt_hip_bapply: nc <= 256, na <= 512 required");
        return RSVDT_HIP_ERR_ARG;
    }
    int ncpad = 1;
    while (ncpad < nc) ncpad <<= 1;
    int rb = 256 / ncpad;
    const int64_t rb_lds = 65536 / ((na > 0 ? na : 1) * 16);
    if (rb > rb_lds) rb = (int)(rb_lds > 0 ? rb_lds : 1);
    const size_t lds = (size_t)rb * (size_t)(na > 0 ? na : 1) * 16;
    hipLaunchKernelGGL(k_bapply, dim3(ceil_div(nrows, rb), (unsigned)nbatch), dim3(256), lds, st, nrows,
                       na, nc, ncpad, rb, (const double2 *)X, xb, xr, xa, (const double2 *)C, alpha,
                       (const double2 *)Y, yb, yr, yc, (double2 *)Out, ob, orow, oc);
    RSVDT_LAUNCH_CHECK("rsvdt_hip_bapply");
    return RSVDT_HIP_OK;
}

// Workgroups per batch: enough for the resident waves of all CUs (four
// workgroups a CU for one column tile, two for two, one above), at most one per
// four row tiles, and at most the partials the Gram's work buffer has room for.
template <int TC, bool GRAM>
static int launch_bapply_gram(int64_t nbatch, int64_t nrows, int64_t n, const double2 *X, int64_t xb, int64_t xr,
                              const double2 *C, double2 *Out, double2 *part, int64_t *nparts, hipStream_t s)
{
    const int64_t ntile = (nrows + (TC == 1 ? 32 : 16) - 1) / (TC == 1 ? 32 : 16);
    int64_t gx = ((TC == 1 ? 1024 : (TC == 2 ? 512 : 256)) + nbatch - 1) / nbatch;
    if (gx > (ntile + 3) / 4) gx = (ntile + 3) / 4;
    const int64_t room = bgram_work_parts(nbatch, nrows, n, n);
    if (GRAM && gx > room) gx = room;
    const size_t lds = (size_t)(256 * TC * TC) * 16;
    const dim3 grid((unsigned)gx, 1, (unsigned)nbatch);
    if ((double)nbatch * (double)nrows * (double)n * 16.0 > 256e6)
        hipLaunchKernelGGL((k_bapply_gram<TC, GRAM, true>), grid, dim3(256), lds, s, nrows, (int)n, X, xb, xr, C, Out,
                           part);
    else
        hipLaunchKernelGGL((k_bapply_gram<TC, GRAM, false>), grid, dim3(256), lds, s, nrows, (int)n, X, xb, xr, C, Out,
                           part);
    RSVDT_LAUNCH_CHECK("rsvdt_hip_bapply_gram");
    *nparts = gx;
    return RSVDT_HIP_OK;
}

extern "C" int rsvdt_hip_bapply_gram(int64_t nbatch, int64_t nrows, int64_t n, const double *X, int64_t xb, int64_t xr,
                                     const double *C, double *Out, double *G, void *work, rsvdt_stream_t s)
{
    if (nbatch <= 0 || nrows <= 0 || n <= 0) return RSVDT_HIP_OK;
    if (nbatch > 65535 || n > 64 || (G && !work)) {
        set_error_msg("rsvdt_hip_bapply_gram: nbatch <= 65535, n <= 64 (and work with G) required");
        return RSVDT_HIP_ERR_ARG;
    }
    hipStream_t st = as_stream(s);
    int64_t np = 0;
    int rc = RSVDT_HIP_ERR_ARG;
    const int TC = (int)((n + 15) / 16);
#define RSVDT_AG(T)                                                                                              \
    if (TC == T)                                                                                                 \
        rc = G ? launch_bapply_gram<T, true>(nbatch, nrows, n, (const double2 *)X, xb, xr, (const double2 *)C,   \
                                             (double2 *)Out, (double2 *)work, &np, st)                           \
               : launch_bapply_gram<T, false>(nbatch, nrows, n, (const double2 *)X, xb, xr, (const double2 *)C,  \
                                              (double2 *)Out, nullptr, &np, st);
    RSVDT_AG(1) RSVDT_AG(2) RSVDT_AG(3)
#undef RSVDT_AG
    if (TC == 4) {          // both accumulator sets do not fit beside the operands: the Gram on its own
        rc = launch_bapply_gram<4, false>(nbatch, nrows, n, (const double2 *)X, xb, xr, (const double2 *)C,
                                          (double2 *)Out, nullptr, &np, st);
        return rc || !G ? rc : rsvdt_hip_bgram(nbatch, nrows, n, n, Out, xb, xr, 1, Out, xb, xr, 1, G, work, s);
    }
    if (rc || !G) return rc;
    hipLaunchKernelGGL(k_bgram_reduce, bgram_reduce_grid(n * n, nbatch), dim3(256), 0, st, np, (int)n, (int)n,
                       1, TC, (const double2 *)work, (double2 *)G);
    RSVDT_LAUNCH_CHECK("rsvdt_hip_bapply_gram(reduce)");
    return RSVDT_HIP_OK;
}

// Measured products, one after another on a stream (N = 32 .. 1860, 1 to 650
// columns): 5 us up to 200 rows, a launch; then 4 rows a workgroup 6.8 us at 500,
// 12.5 at 1000; 16 rows 8.1 us at 500, 14 at 1000, 24 at 1860 for each round of as
// many workgroups as CUs, and 11, 19, 35 us with two column tiles.
extern "C" double rsvdt_hip_dense_apply_us(int64_t N, int64_t cols)
{
    const double n = (double)N, least = 5.0;
    if (cols <= 16 && N <= 1024) return n < 240 ? least : 2.5 + 0.0105 * n;
    const int64_t ct = cols <= 256 ? 16 : 32, wg = ((N + 15) / 16) * ((cols + ct - 1) / ct), cus = device_cus();
    const double one = cols <= 256 ? 2.0 + 0.012 * n : 2.0 + 0.018 * n;
    return (one < least ? least : one) * (double)((wg + cus - 1) / cus);
}

extern "C" int rsvdt_hip_dense_apply(int64_t N, int64_t k, int64_t nb, const double *E, const double *X,
                                     const double *F, double *Out, rsvdt_stream_t s)
{
    if (N <= 0 || k <= 0 || nb <= 0) return RSVDT_HIP_OK;
    if (N > 65536 || k * nb > 65535LL * 16 || X == Out) {
        set_error_msg("rsvdt_hip_dense_apply: N <= 65536, at most 16 x 65535 columns, out of place");
        return RSVDT_HIP_ERR_ARG;
    }
    const int ncol = (int)(k * nb);
    // one column tile: 16 rows a workgroup would leave most CUs idle (us, 16 and 4
    // rows: N = 300 7.7, 6.7; 500 7.8, 6.6; 700 10.5, 8.5; 1000 13.3, 12.6); with
    // more column tiles the rows of X that every workgroup reads cost more (N =
    // 500, 33 columns: 8.0, 10.4)
    if (ncol <= 16 && N <= 1024)
        hipLaunchKernelGGL((k_dense_apply<1, 4>), dim3(ceil_div(N, 4)), dim3(512), 0, as_stream(s), (int)N, (int)k, ncol,
                           (const double2 *)E, (const double2 *)X, (const double2 *)F, (double2 *)Out);
    else if (ncol <= 256)
        hipLaunchKernelGGL((k_dense_apply<1, 16>), dim3(ceil_div(N, 16), ceil_div(ncol, 16)), dim3(512), 0, as_stream(s), (int)N,
                           (int)k, ncol, (const double2 *)E, (const double2 *)X, (const double2 *)F, (double2 *)Out);
    else
        hipLaunchKernelGGL((k_dense_apply<2, 16>), dim3(ceil_div(N, 16), ceil_div(ncol, 32)), dim3(512), 0, as_stream(s), (int)N,
                           (int)k, ncol, (const double2 *)E, (const double2 *)X, (const double2 *)F, (double2 *)Out);
    RSVDT_LAUNCH_CHECK("rsvdt_hip_dense_apply");
    return RSVDT_HIP_OK;
}
