// hv_s12.hip -- S=1/2 matrix-free H.v for gfx950 (CDNA4).
//
// Computes the reference's p_mltply_v3 (S_one_half/Hybrid_TPS_parallel.f90:190-263):
//     v0 += (H - ibond*eperbd) v1,   prdct = <v1|(H - ibond*eperbd)|v1>
// with H given by the bond matrices of H_dot_v (same file, 305-442).  Instead of the
// reference's 4*ibond full passes over the vector, the host planner (context.cpp)
// rewrites H as a diagonal D(i) plus flip terms  c_t(sel(i)) * v1(i ^ mask_t)  and groups
// the terms into a few "tile passes".  A pass picks K memory-index bits (the tile bits);
// every term of the pass flips only tile bits, so a workgroup that stages one tile
// (2^K consecutive-in-tile states, strided in memory over the non-tile bits) in LDS
// can apply all of the pass's terms without touching HBM again.  Each pass reads v1
// once and read-modify-writes v0 once.
//
// Memory index m = (state << colbits) | column: batched vectors ([dim][nvec] interleaved)
// add never-flipped column bits at the bottom, which the planner keeps in the tile so
// the 16-byte lanes of a wave form contiguous runs.
#include <cstring>
#include <mutex>
#include <utility>

#include "internal.h"

namespace pned {

struct PassArgs {
    uint64_t tile_count;   // number of tiles = 2^(outer bits)
    int K;                 // tile bits
    int nouter;
    int colbits;
    int first_term, nterm;
    int diag;              // add the diagonal (first pass)
    int fresh;             // first pass: v0 input is zero
    int ncol;              // columns (1 << colbits)
    int nlo;               // outer bits resolved by the first base table
    int nop;               // >1: one operator per column (batch context)
    double shift;          // -ibond * eperbd, added to the diagonal
    const double *colcoef; // [devterm][nop][4] when nop > 1
    const double *coldiag; // [nop][ngroups+1][2] when nop > 1
    const double *colscale;// per-column factor on v1 (H (s v1)); null = 1
    const double *yscale;  // diagonal pass: per-column factor on the v0 input (v0 = y v0 + ...); null = 1
    int ncat[4];           // term-major kernel: terms per category (see build_tm_terms)
    int ngroups;           // diagonal groups (batch contexts stage their weights)
    // term-major kernel, last pass of a deferred-normalisation Lanczos step:
    //   1  only the <v1|H_pass v1> partials (no v0 traffic)
    //   2  v0 := w - Re(alpha) s v1 with w = v0 + H_pass (s v1), alpha = s * lz_prd[c],
    //      partials [|w - alpha s v1|^2, 0]
    int lz_mode;
    const double *lz_prd;
    int nt;                // term-major kernel: NT_V1 / NT_V0 streams
};

// Per-pass address tables in device memory (read with scalar loads):
//   lo[t]  memory-index offset of thread t's slot (tile bits 0..LT-1)
//   hi[r]  offset of register slot r (tile bits LT..K-1)
//   blo/bhi  tile base = blo[tix & (2^nlo - 1)] | bhi[tix >> nlo]  (outer bits)
constexpr int PD_LO = 1024, PD_HI = 32, PD_B = 2048;
struct PassDev {
    uint64_t lo[PD_LO];
    uint64_t hi[PD_HI];
    uint64_t blo[PD_B];
    uint64_t bhi[PD_B];
};

template <typename R> struct C2;
template <> struct C2<double> { using T = double2; };
template <> struct C2<float> { using T = float2; };

// vector elements with a non-temporal hint (streams that the caches should not keep)
template <typename V>
__device__ __forceinline__ V ld_nt(const V *p)
{
    using X = decltype(V::x) __attribute__((ext_vector_type(2)));
    const X t = __builtin_nontemporal_load(reinterpret_cast<const X *>(p));
    V v;
    v.x = t.x;
    v.y = t.y;
    return v;
}
template <typename V>
__device__ __forceinline__ void st_nt(V *p, const V &v)
{
    using X = decltype(V::x) __attribute__((ext_vector_type(2)));
    X t;
    t.x = v.x;
    t.y = v.y;
    __builtin_nontemporal_store(t, reinterpret_cast<X *>(p));
}

__device__ __forceinline__ double diag_value_re(const DiagDev &d, uint32_t s, double &im)
{
    double re = d.c0r;
    im = d.c0i;
    for (int g = 0; g < d.ngroups; ++g) {
        uint32_t f = (d.kind[g] == 0) ? (s & d.mask[g]) : ((s ^ (s >> d.shift[g])) & d.mask[g]);
        const double c = (double)__popc(f);
        re = fma(c, d.wr[g], re);
        im = fma(c, d.wi[g], im);
    }
    return re;
}

template <int... Is, typename F>
__device__ __forceinline__ void static_for_impl(std::integer_sequence<int, Is...>, F &&f)
{
    (f(std::integral_constant<int, Is>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F &&f)
{
    static_for_impl(std::make_integer_sequence<int, N>{}, f);
}

// a wave-uniform double held in scalar registers
__device__ __forceinline__ double uniform(double v)
{
    const uint64_t u = (uint64_t)__double_as_longlong(v);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)u);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(u >> 32));
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

// TPB threads, R states per thread: tile of K = log2(TPB*R) bits.  Tile slot
// j = tid + TPB*r holds the state with memory index base | offLo(tid) | offHi(r).
// Software pipeline over the tiles a block owns: while tile t is computed from LDS, the
// v1 values of tile t+1 are in flight into registers (written to LDS after the barrier
// that ends tile t), and the v0 values being accumulated arrive one chunk of CH states
// ahead of their use, across tile boundaries.  HBM latency is hidden inside one
// workgroup, which matters when a 128 KB tile leaves room for one workgroup per CU.
template <typename Real, int TPB, int R>
__global__ __launch_bounds__(TPB) void hv_s12_pass(const typename C2<Real>::T *__restrict__ v1,
                                                   typename C2<Real>::T *__restrict__ v0,
                                                   const DevTerm *__restrict__ terms,
                                                   const DiagDev *__restrict__ diagp,
                                                   const PassDev *__restrict__ pd, PassArgs a,
                                                   double *__restrict__ partial)
{
    using V = typename C2<Real>::T;
    extern __shared__ unsigned char smem_raw[];
    V *tile = reinterpret_cast<V *>(smem_raw);
    const unsigned char *tbytes = smem_raw;  // partner slot j ^ m sits at byte (16 j) ^ (16 m)
    constexpr int CH = (R < 4) ? R : 4;      // states per compute chunk
    constexpr int NCH = R / CH;
    const int tid = threadIdx.x;

    const uint64_t offLo = pd->lo[tid];
    auto offHi = [&](int r) { return pd->hi[r]; };
    const bool rd0 = !(a.diag && a.fresh);
    const double ys = (a.diag && a.yscale) ? a.yscale[tid & (a.ncol - 1)] : 1.0;
    const uint64_t lomask = (1ull << a.nlo) - 1;
    auto tile_base = [&](uint64_t tix) { return pd->blo[tix & lomask] | pd->bhi[tix >> a.nlo] | offLo; };

    double pr_re = 0.0, pr_im = 0.0;
    // prefetch registers kept as scalar components (a V[] array is not promoted to
    // registers for the 16-byte type)
    Real xr_[R], xi_[R];
    Real ycr[CH], yci[CH];
    auto fetch_x = [&](uint64_t b) {
        static_for<R>([&](auto I) {
            const V t = v1[b | offHi(I)];
            xr_[I] = t.x;
            xi_[I] = t.y;
        });
    };
    uint64_t tix = blockIdx.x;
    if (tix < a.tile_count) {
        const uint64_t tb0 = tile_base(tix);
        fetch_x(tb0);
        if (rd0) static_for<CH>([&](auto I) { const V t = v0[tb0 | offHi(I)]; ycr[I] = t.x; yci[I] = t.y; });
    }
    for (; tix < a.tile_count; tix += gridDim.x) {
        const uint64_t tb0 = tile_base(tix);
        static_for<R>([&](auto I) {
            V t;
            t.x = xr_[I];
            t.y = xi_[I];
            tile[tid + TPB * I] = t;
        });
        __syncthreads();
        const uint64_t nx = tix + gridDim.x;
        const bool has_next = nx < a.tile_count;
        const uint64_t nb = has_next ? tile_base(nx) : 0;
        if (has_next) fetch_x(nb);

        static_for<NCH>([&](auto CI) {
            constexpr int r0 = CI * CH;
            // v0 of the next chunk (or of the next tile's first chunk)
            Real ynr[CH], yni[CH];
            if (rd0) {
                if constexpr (r0 + CH < R) {
                    static_for<CH>([&](auto I) {
                        const V t = v0[tb0 | offHi(r0 + CH + I)];
                        ynr[I] = t.x;
                        yni[I] = t.y;
                    });
                } else {
                    if (has_next)
                        static_for<CH>([&](auto I) {
                            const V t = v0[nb | offHi(I)];
                            ynr[I] = t.x;
                            yni[I] = t.y;
                        });
                }
            }
            uint32_t st[CH], jb[CH];
            double ar[CH], ai[CH];
            static_for<CH>([&](auto c) {
                jb[c] = (uint32_t)((tid + TPB * (r0 + c)) * sizeof(V));   // LDS byte offset of the slot
                st[c] = (uint32_t)((tb0 | offHi(r0 + c)) >> a.colbits);
                ar[c] = 0.0;
                ai[c] = 0.0;
            });
            if (a.diag) {
                const DiagDev &dg = *diagp;
                static_for<CH>([&](auto c) {
                    double di, dr;
                    if (a.nop > 1) {
                        // per-column weights; the thread's column is tid & (nop-1)
                        const double *w = a.coldiag + (size_t)(tid & (a.nop - 1)) * (dg.ngroups + 1) * 2;
                        dr = w[2 * dg.ngroups];
                        di = w[2 * dg.ngroups + 1];
                        for (int g = 0; g < dg.ngroups; ++g) {
                            const uint32_t f = (dg.kind[g] == 0) ? (st[c] & dg.mask[g])
                                                                 : ((st[c] ^ (st[c] >> dg.shift[g])) & dg.mask[g]);
                            const double cnt = (double)__popc(f);
                            dr = fma(cnt, w[2 * g], dr);
                            di = fma(cnt, w[2 * g + 1], di);
                        }
                        dr += a.shift;
                    } else {
                        dr = diag_value_re(dg, st[c], di) + a.shift;
                    }
                    const V x = tile[tid + TPB * (r0 + c)];
                    ar[c] = dr * (double)x.x - di * (double)x.y;
                    ai[c] = dr * (double)x.y + di * (double)x.x;
                });
            }
            if (a.nop > 1) {
                const double *cbase = a.colcoef + (size_t)(tid & (a.nop - 1)) * 4;
                for (int t = 0; t < a.nterm; ++t) {
                    const DevTerm T = terms[a.first_term + t];
                    const double *cc = cbase + (size_t)(a.first_term + t) * a.nop * 4;
                    const double c0r = cc[0], c0i = cc[1];
                    const double dr = cc[2] - c0r, di = cc[3] - c0i;
                    const uint32_t tmb = T.tmask * (uint32_t)sizeof(V);
                    static_for<CH>([&](auto c) {
                        const V p = *reinterpret_cast<const V *>(tbytes + (jb[c] ^ tmb));
                        const double sel = (double)(__popc(st[c] & T.selmask) & 1);
                        const double cr = fma(sel, dr, c0r), ci = fma(sel, di, c0i);
                        ar[c] = fma(cr, (double)p.x, ar[c]);
                        ar[c] = fma(-ci, (double)p.y, ar[c]);
                        ai[c] = fma(cr, (double)p.y, ai[c]);
                        ai[c] = fma(ci, (double)p.x, ai[c]);
                    });
                }
            } else
            for (int t = 0; t < a.nterm; ++t) {
                const DevTerm T = terms[a.first_term + t];
                if (T.is_real) {
                    const double d = T.c1r - T.c0r;
                    const uint32_t tmb = T.tmask * (uint32_t)sizeof(V);
                    static_for<CH>([&](auto c) {
                        const V p = *reinterpret_cast<const V *>(tbytes + (jb[c] ^ tmb));
                        const double sel = (double)(__popc(st[c] & T.selmask) & 1);
                        const double cf = fma(sel, d, T.c0r);
                        ar[c] = fma(cf, (double)p.x, ar[c]);
                        ai[c] = fma(cf, (double)p.y, ai[c]);
                    });
                } else {
                    const double dr = T.c1r - T.c0r, di = T.c1i - T.c0i;
                    const uint32_t tmb = T.tmask * (uint32_t)sizeof(V);
                    static_for<CH>([&](auto c) {
                        const V p = *reinterpret_cast<const V *>(tbytes + (jb[c] ^ tmb));
                        const double sel = (double)(__popc(st[c] & T.selmask) & 1);
                        const double cr = fma(sel, dr, T.c0r), ci = fma(sel, di, T.c0i);
                        ar[c] = fma(cr, (double)p.x, ar[c]);
                        ar[c] = fma(-ci, (double)p.y, ar[c]);
                        ai[c] = fma(cr, (double)p.y, ai[c]);
                        ai[c] = fma(ci, (double)p.x, ai[c]);
                    });
                }
            }
            if (a.colscale) {
                const double sc = a.colscale[tid & (a.ncol - 1)];
                static_for<CH>([&](auto c) {
                    ar[c] *= sc;
                    ai[c] *= sc;
                });
            }
            static_for<CH>([&](auto c) {
                const V x = tile[tid + TPB * (r0 + c)];
                pr_re += (double)x.x * ar[c] + (double)x.y * ai[c];
                pr_im += (double)x.x * ai[c] - (double)x.y * ar[c];
                V o;
                if (rd0) {
                    o.x = (Real)fma(ys, (double)ycr[c], ar[c]);
                    o.y = (Real)fma(ys, (double)yci[c], ai[c]);
                } else {
                    o.x = (Real)ar[c];
                    o.y = (Real)ai[c];
                }
                v0[tb0 | offHi(r0 + c)] = o;
            });
            if (rd0) static_for<CH>([&](auto I) { ycr[I] = ynr[I]; yci[I] = yni[I]; });
        });
        __syncthreads();
    }

    // deterministic block reduction per column: lanes with equal (tid & (ncol-1)) belong to
    // the same column (the planner keeps the column bits as the lowest tile bits)
    double *red = reinterpret_cast<double *>(smem_raw);
    red[2 * tid] = pr_re;
    red[2 * tid + 1] = pr_im;
    __syncthreads();
    for (int s = TPB / 2; s >= a.ncol && s > 0; s >>= 1) {
        if (tid < s) {
            red[2 * tid] += red[2 * (tid + s)];
            red[2 * tid + 1] += red[2 * (tid + s) + 1];
        }
        __syncthreads();
    }
    if (tid < a.ncol) {
        partial[(size_t)blockIdx.x * 2 * a.ncol + 2 * tid] = red[2 * tid];
        partial[(size_t)blockIdx.x * 2 * a.ncol + 2 * tid + 1] = red[2 * tid + 1];
    }
}

// Term-major pass kernel.  Same tiles, tables and results as hv_s12_pass, but the loop
// runs over terms outside and over register slots of a thread inside, with one
// accumulator per slot.  For a term with flip mask m and selector mask s (tile slot
// j = tid + TPB r):
//   partner slot  j ^ m = (tid ^ m_lo) + TPB (r ^ m_hi)
//   selector      parity(tid & s_lo) ^ parity(outer & s_out) ^ parity(r & s_hi)
// The first two parts are fixed for the (thread, tile): they pick the two coefficients
// once per term per sweep; the register part is uniform across the wave.  A state-term
// then costs one address add, one LDS read and 2 (real) or 4 (complex) FMAs, plus a
// 64-bit select for terms whose selector has register bits.  The host sorts each pass's
// terms into these four categories so every category is one straight-line loop (the
// accumulators never pass through divergent merges).
//
// The R slots of a tile are accumulated in R/S sweeps of S slots, so only S accumulators
// and S v0 values are live next to the R prefetched v1 values of the next tile; a sweep's
// v0 values are in flight while its terms are applied.  Accumulates in Real (FP64 for complex128, FP32 for complex64
// storage); the <x|Hx> partials are FP64.
//
// Non-temporal streams (nt): where the two vectors together exceed the 256 MB Infinity Cache, v0
// is read and written with the non-temporal hint, and v1 as well where it alone exceeds it, so
// a v1 that fits is still there when the next pass reads it (N=24 with field, complex128: 605 ->
// 565 us at 1024 threads; N=28 9.40 -> 9.08 ms, N=30 45.4 -> 45.0 ms; complex64 runs of 64 bytes
// lose, 5.80 -> 6.48 ms at N=28, because a line's other half is fetched again).
//
// 2^12-state complex128 tiles on 512 threads are held to 128 VGPRs (sweeps of 4 slots): two
// blocks then share a CU (64 KB of LDS each) and one's loads run under the other's barriers
// (N=24 with field: 677 -> 533 us per H.v; one 1024-thread block per CU 565 us).
template <typename Real, int TPB, int R>
constexpr int TM_WAVES = (sizeof(Real) == 8 && TPB == 512 && R == 8) ? 4 : 1;
template <typename Real, int TPB, int R, int S>
__global__ __launch_bounds__(TPB, (TM_WAVES<Real, TPB, R>)) void hv_s12_tm(const typename C2<Real>::T *__restrict__ v1,
                                                 typename C2<Real>::T *__restrict__ v0,
                                                 const TmTerm *__restrict__ terms,
                                                 const DiagDev *__restrict__ diagp,
                                                 const PassDev *__restrict__ pd, PassArgs a,
                                                 double *__restrict__ partial)
{
    static_assert(R % S == 0, "sweeps must tile the register slots");
    using V = typename C2<Real>::T;
    using A = Real;
    constexpr int NS = R / S;
    extern __shared__ unsigned char smem_raw[];
    V *tile = reinterpret_cast<V *>(smem_raw);
    const int tid = threadIdx.x;
    const uint64_t offLo = pd->lo[tid];
    const bool rd0 = !(a.diag && a.fresh) && a.lz_mode != 1;
    const uint64_t lomask = (1ull << a.nlo) - 1;
    auto outer_base = [&](uint64_t tix) { return pd->blo[tix & lomask] | pd->bhi[tix >> a.nlo]; };
    constexpr uint32_t RSTRIDE = (uint32_t)(TPB * sizeof(V));   // bytes between register slots
    const uint32_t lane_b = (uint32_t)tid * (uint32_t)sizeof(V);

    // batch contexts: this pass's per-column coefficients [term][column][4] and, in the
    // diagonal pass, the per-column diagonal weights [column][groups+1][2], after the tile
    double *ccol = reinterpret_cast<double *>(smem_raw + sizeof(V) * TPB * R);
    double *cdiag = ccol + (a.nop > 1 ? (size_t)a.nterm * a.nop * 4 : 0);
    if (a.nop > 1) {
        const int n = a.nterm * a.nop * 4;
        const double *src = a.colcoef + (size_t)a.first_term * a.nop * 4;
        for (int i = tid; i < n; i += TPB) ccol[i] = src[i];
        if (a.diag)
            for (int i = tid; i < a.nop * (a.ngroups + 1) * 2; i += TPB) cdiag[i] = a.coldiag[i];
    }
    const A colsc = a.colscale ? (A)a.colscale[tid & (a.ncol - 1)] : (A)1;
    const A ys = (a.diag && a.yscale) ? (A)a.yscale[tid & (a.ncol - 1)] : (A)1;
    double lar = 0.0, lai = 0.0;
    if (a.lz_mode == 2) {
        lar = (double)colsc * a.lz_prd[2 * (tid & (a.ncol - 1))];
        lai = (double)colsc * a.lz_prd[2 * (tid & (a.ncol - 1)) + 1];
    }

    // the diagonal as a lane program (see DiagDev): group e in lane e, class weights in
    // lanes 48..63; one operator only (batch contexts weight per column)
    const int dprog = (a.diag && a.nop <= 1) ? diagp->nprog : 0;
    const int drest = dprog ? diagp->nrest : 0;   // split program: lanes dprog.. counted per tile
    const uint32_t dpa = dprog ? diagp->prog_a[tid & 63] : 0u;
    const uint32_t dpb = dprog ? diagp->prog_b[tid & 63] : 0u;

    double pr_re = 0.0, pr_im = 0.0;
    Real xr[R], xi[R];
    const bool nt1 = a.nt & NT_V1, nt0 = a.nt & NT_V0;
    auto fetch_x = [&](uint64_t b) {
        if (nt1)
            static_for<R>([&](auto I) {
                const V t = ld_nt(&v1[b | pd->hi[I]]);
                xr[I] = t.x;
                xi[I] = t.y;
            });
        else
            static_for<R>([&](auto I) {
                const V t = v1[b | pd->hi[I]];
                xr[I] = t.x;
                xi[I] = t.y;
            });
    };
    auto fetch_y = [&](uint64_t b, int r0, Real *yr, Real *yi) {
        if (nt0)
            static_for<S>([&](auto I) {
                const V t = ld_nt(&v0[b | pd->hi[r0 + I]]);
                yr[I] = t.x;
                yi[I] = t.y;
            });
        else
            static_for<S>([&](auto I) {
                const V t = v0[b | pd->hi[r0 + I]];
                yr[I] = t.x;
                yi[I] = t.y;
            });
    };
    // each block takes a contiguous range of tiles: consecutive tiles of a block differ in the
    // lowest outer bits, so its runs follow each other in memory (measured at N=32: a few per
    // cent on the passes whose tiles hold few low memory bits, against tiles strided by the grid)
    const uint64_t per = (a.tile_count + gridDim.x - 1) / gridDim.x;
    uint64_t tix = (uint64_t)blockIdx.x * per;
    const uint64_t tend = (tix + per < a.tile_count) ? tix + per : a.tile_count;
    if (tix < tend) fetch_x(outer_base(tix) | offLo);
    for (; tix < tend; ++tix) {
        const uint64_t ob = outer_base(tix);
        const uint64_t tb0 = ob | offLo;
        static_for<R>([&](auto I) {
            V t;
            t.x = xr[I];
            t.y = xi[I];
            tile[tid + TPB * I] = t;
        });
        __syncthreads();
        // v0 of the first sweep goes out before the next tile's v1, so waiting for it does
        // not wait for the prefetch (vector memory counters retire in order)
        Real ycr[S], yci[S];
        if (rd0) fetch_y(tb0, 0, ycr, yci);
        const uint64_t nx = tix + 1;
        if (nx < tend) fetch_x(outer_base(nx) | offLo);
        // the diagonal's per-class counts over the bit positions that no register bit takes
        // part in: the same for every slot of this thread and tile (16 bits per class)
        uint64_t rcnt = 0;
        if (drest) {
            const uint32_t s0 = (uint32_t)(tb0 >> a.colbits);
            uint32_t acc = 0;
            for (int e = dprog; e < dprog + drest; ++e) {
                const uint32_t pa = (uint32_t)__builtin_amdgcn_readlane((int)dpa, e);
                const uint32_t m = (uint32_t)__builtin_amdgcn_readlane((int)dpb, e);
                acc += (uint32_t)__popc(((pa & 64u) ? (s0 ^ (s0 >> (pa & 63u))) : s0) & m);
                if (pa & 128u) {
                    rcnt |= (uint64_t)acc << (16u * ((pa >> 8) & 7u));
                    acc = 0u;
                }
            }
        }

        static_for<NS>([&](auto HI) {
            constexpr int r0 = HI * S;
            if constexpr (r0 > 0) {
                if (rd0) fetch_y(tb0, r0, ycr, yci);
            }
            A ar[S], ai[S];
            if (dprog) {
                // all S slots at once, group-outer: per group two readlanes, per slot a shift,
                // an xor and an and with a popcount; per weight class one convert and FMA pair
                // a slot's state is sb | hs[I] (disjoint bits), and x -> x ^ (x >> sh) is linear
                // over xor, so a group's bits of slot I are its bits of sb (per thread, formed
                // once per group) xor those of hs[I] (uniform, on the scalar unit)
                uint32_t cnt[S], hs[S];
                double dr[S], di[S];
                const double d0r = diagp->c0r + a.shift, d0i = diagp->c0i;
                const uint32_t sb = (uint32_t)(tb0 >> a.colbits);
                static_for<S>([&](auto I) {
                    hs[I] = (uint32_t)(pd->hi[r0 + I] >> a.colbits);
                    cnt[I] = 0u;
                    dr[I] = d0r;
                    di[I] = d0i;
                });
                for (int e = 0; e < dprog; ++e) {
                    const uint32_t pa = (uint32_t)__builtin_amdgcn_readlane((int)dpa, e);
                    const uint32_t m = (uint32_t)__builtin_amdgcn_readlane((int)dpb, e);
                    const uint32_t sh = pa & 63u;
                    if (pa & 64u) {
                        const uint32_t f = (sb ^ (sb >> sh)) & m;
                        static_for<S>([&](auto I) {
                            cnt[I] += (uint32_t)__popc(f ^ ((hs[I] ^ (hs[I] >> sh)) & m));
                        });
                    } else {
                        const uint32_t f = sb & m;
                        static_for<S>([&](auto I) { cnt[I] += (uint32_t)__popc(f ^ (hs[I] & m)); });
                    }
                    if (pa & 128u) {
                        const int c = (int)((pa >> 8) & 7u);
                        const uint32_t rc = (uint32_t)(rcnt >> (16 * c)) & 0xFFFFu;
                        const uint64_t wrb = (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)dpa, 48 + c) |
                                             ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)dpa, 56 + c) << 32);
                        const uint64_t wib = (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)dpb, 48 + c) |
                                             ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)dpb, 56 + c) << 32);
                        const double wr = __longlong_as_double((long long)wrb);
                        const double wi = __longlong_as_double((long long)wib);
                        static_for<S>([&](auto I) {
                            dr[I] = fma((double)(cnt[I] + rc), wr, dr[I]);
                            di[I] = fma((double)(cnt[I] + rc), wi, di[I]);
                            cnt[I] = 0u;
                        });
                    }
                }
                static_for<S>([&](auto I) {
                    const V x = tile[tid + TPB * (r0 + I)];
                    ar[I] = (A)(dr[I] * (double)x.x - di[I] * (double)x.y);
                    ai[I] = (A)(dr[I] * (double)x.y + di[I] * (double)x.x);
                });
            } else if (a.diag) {
                const DiagDev &dg = *diagp;
                static_for<S>([&](auto I) {
                    const uint32_t st = (uint32_t)((tb0 | pd->hi[r0 + I]) >> a.colbits);
                    double dr, di;
                    if (a.nop > 1) {
                        const double *w = cdiag + (size_t)(tid & (a.nop - 1)) * (dg.ngroups + 1) * 2;
                        dr = w[2 * dg.ngroups];
                        di = w[2 * dg.ngroups + 1];
                        for (int g = 0; g < dg.ngroups; ++g) {
                            const uint32_t f = (dg.kind[g] == 0) ? (st & dg.mask[g])
                                                                 : ((st ^ (st >> dg.shift[g])) & dg.mask[g]);
                            const double cnt = (double)__popc(f);
                            dr = fma(cnt, w[2 * g], dr);
                            di = fma(cnt, w[2 * g + 1], di);
                        }
                        dr += a.shift;
                    } else {
                        dr = diag_value_re(dg, st, di) + a.shift;
                    }
                    const V x = tile[tid + TPB * (r0 + I)];
                    ar[I] = (A)(dr * (double)x.x - di * (double)x.y);
                    ai[I] = (A)(dr * (double)x.y + di * (double)x.x);
                });
            } else {
                static_for<S>([&](auto I) {
                    ar[I] = (A)0;
                    ai[I] = (A)0;
                });
            }

            // terms come sorted by category: [real | real, register selector | complex |
            // complex, register selector]; one straight-line loop per category
            int t = a.first_term;
            auto prelude = [&](const TmTerm &T, A &car, A &cai, A &cbr, A &cbi) {
                const uint32_t par = (uint32_t)(__popc((uint32_t)tid & T.slo) + __popcll(ob & T.sout)) & 1u;
                A c0r, c0i, c1r, c1i;
                if (a.nop > 1) {
                    // per-column coefficients, staged in LDS for this pass
                    const double *cc =
                        ccol + ((size_t)(T.term - a.first_term) * a.nop + (size_t)(tid & (a.nop - 1))) * 4;
                    c0r = (A)cc[0];
                    c0i = (A)cc[1];
                    c1r = (A)cc[2];
                    c1i = (A)cc[3];
                } else {
                    // uniform: kept in scalar registers (a per-lane select of two loaded
                    // values would otherwise become a per-lane load)
                    c0r = (A)uniform(T.c0r);
                    c0i = (A)uniform(T.c0i);
                    c1r = (A)uniform(T.c1r);
                    c1i = (A)uniform(T.c1i);
                }
                car = par ? c1r : c0r;   // coefficient where the register part of the selector is even
                cai = par ? c1i : c0i;
                cbr = par ? c0r : c1r;   // ... and where it is odd
                cbi = par ? c0i : c1i;
                return smem_raw + (lane_b ^ (T.mlo * (uint32_t)sizeof(V)));
            };
            constexpr int G = (S < 4) ? S : 4;   // partner reads issued ahead of their FMAs
            auto run_cat = [&](int count, auto CXc, auto SELc) {
                constexpr bool CX = decltype(CXc)::value;
                constexpr bool SEL = decltype(SELc)::value;
                for (const int e = t + count; t < e; ++t) {
                    const TmTerm T = terms[t];
                    A car, cai, cbr, cbi;
                    const unsigned char *lb = prelude(T, car, cai, cbr, cbi);
                    static_for<S / G>([&](auto GI) {
                        Real qr[G], qi[G];
                        static_for<G>([&](auto k) {
                            constexpr int r = r0 + GI * G + k;
                            const V p = *reinterpret_cast<const V *>(lb + ((uint32_t)r ^ T.mhi) * RSTRIDE);
                            qr[k] = p.x;
                            qi[k] = p.y;
                        });
                        static_for<G>([&](auto k) {
                            constexpr int r = r0 + GI * G + k;
                            constexpr int u = GI * G + k;
                            A cr = car, ci = cai;
                            if constexpr (SEL) {
                                const bool f = __popc((uint32_t)r & T.shi) & 1;
                                cr = f ? cbr : car;
                                if constexpr (CX) ci = f ? cbi : cai;
                            }
                            if constexpr (CX) {
                                ar[u] = fma(cr, (A)qr[k], ar[u]);
                                ar[u] = fma(-ci, (A)qi[k], ar[u]);
                                ai[u] = fma(cr, (A)qi[k], ai[u]);
                                ai[u] = fma(ci, (A)qr[k], ai[u]);
                            } else {
                                ar[u] = fma(cr, (A)qr[k], ar[u]);
                                ai[u] = fma(cr, (A)qi[k], ai[u]);
                            }
                        });
                    });
                }
            };
            run_cat(a.ncat[0], std::false_type{}, std::false_type{});
            run_cat(a.ncat[1], std::false_type{}, std::true_type{});
            run_cat(a.ncat[2], std::true_type{}, std::false_type{});
            run_cat(a.ncat[3], std::true_type{}, std::true_type{});

            if (a.colscale) {
                static_for<S>([&](auto I) {
                    ar[I] *= colsc;
                    ai[I] *= colsc;
                });
            }
            // ar, ai become the values to store (nothing is stored in lz_mode 1)
            static_for<S>([&](auto I) {
                const V x = tile[tid + TPB * (r0 + I)];
                if (a.lz_mode == 2) {
                    const double wr0 = (double)fma(ys, (A)ycr[I], ar[I]);
                    const double wi0 = (double)fma(ys, (A)yci[I], ai[I]);
                    const double xr_ = (double)x.x * (double)colsc, xi_ = (double)x.y * (double)colsc;
                    const double wr = wr0 - (lar * xr_ - lai * xi_);
                    const double wi = wi0 - (lar * xi_ + lai * xr_);
                    pr_re = fma(wr, wr, fma(wi, wi, pr_re));
                    ar[I] = (A)(wr0 - lar * xr_);
                    ai[I] = (A)(wi0 - lar * xi_);
                } else {
                    const double hr = (double)ar[I], hi = (double)ai[I];
                    pr_re += (double)x.x * hr + (double)x.y * hi;
                    pr_im += (double)x.x * hi - (double)x.y * hr;
                    if (rd0) {
                        ar[I] = fma(ys, (A)ycr[I], ar[I]);
                        ai[I] = fma(ys, (A)yci[I], ai[I]);
                    }
                }
            });
            auto value = [&](auto I) {
                V o;
                o.x = (Real)ar[I];
                o.y = (Real)ai[I];
                return o;
            };
            if (a.lz_mode != 1) {
                if (nt0)
                    static_for<S>([&](auto I) { st_nt(&v0[tb0 | pd->hi[r0 + I]], value(I)); });
                else
                    static_for<S>([&](auto I) { v0[tb0 | pd->hi[r0 + I]] = value(I); });
            }
        });
        __syncthreads();
    }

    double *red = reinterpret_cast<double *>(smem_raw);
    red[2 * tid] = pr_re;
    red[2 * tid + 1] = pr_im;
    __syncthreads();
    for (int s = TPB / 2; s >= a.ncol && s > 0; s >>= 1) {
        if (tid < s) {
            red[2 * tid] += red[2 * (tid + s)];
            red[2 * tid + 1] += red[2 * (tid + s) + 1];
        }
        __syncthreads();
    }
    if (tid < a.ncol) {
        partial[(size_t)blockIdx.x * 2 * a.ncol + 2 * tid] = red[2 * tid];
        partial[(size_t)blockIdx.x * 2 * a.ncol + 2 * tid + 1] = red[2 * tid + 1];
    }
}

// Short vectors: several workgroups per tile.  A pass of hv_s12_tm on a vector of a few tiles leaves
// most of the chip idle and is one serial chain per tile (address tables, v1, LDS, a scalar-cache
// miss and an LDS round trip per term and sweep, v0, the reduction).  Here every one of a tile's
// `split` workgroups stages the whole tile in LDS and forms one state per thread: the states whose
// low bits in the tile are the workgroup's number.  Addresses come from the bit positions in the
// kernel arguments, v0 is loaded beside v1, and every term record is touched once while those
// loads fly, so the term loop hits the scalar cache.  The states' values are those of hv_s12_tm and
// so are the partial sums: 256 threads owning the tile would each sum their slots and then add in
// halves from the top; a workgroup's states are whole such threads, equal in their low bits, so it
// ends with the first halvings and reduce_split does the rest.
// us per H.v with its reduction and read-back, hv_s12_tm on 256 threads -> here (field, complex128):
// N=12 46.6 -> 30.0, N=16 43.5 -> 37.9, N=18 67 -> 59; 40 Lanczos steps at N=16 2.40 -> 2.02 ms.
constexpr int SPLIT_ROUND = 8;
struct SmallArgs {
    int colbits, ncol;
    int first_term, nreal, nterm;
    int diag, fresh, lz_mode;
    int K, lsplit;         // tile bits, log2 of the workgroups per tile
    double shift;
    const double *colscale, *yscale, *lz_prd;
    uint64_t tb, tbt, tbh; // memory bits of the tile from its bit 0, lsplit and K - lsplit, 5 bits each
    uint64_t ob;           // (an array would be indexed through scratch memory); of the tile number
};

template <typename Real>
__global__ __launch_bounds__(1024) void hv_s12_split(const typename C2<Real>::T *__restrict__ v1,
                                                     typename C2<Real>::T *__restrict__ v0,
                                                     const TmTerm *__restrict__ terms,
                                                     const DiagDev *__restrict__ diagp, SmallArgs a,
                                                     double *__restrict__ partial)
{
    using V = typename C2<Real>::T;
    using A = Real;
    extern __shared__ unsigned char smem_raw[];
    V *tile = reinterpret_cast<V *>(smem_raw);
    const int tid = threadIdx.x, tpb = blockDim.x;   // tpb << lsplit = 2^K
    const uint32_t sub = blockIdx.x & ((1u << a.lsplit) - 1u), tno = blockIdx.x >> a.lsplit;
    // bit k of v to the k-th position (at most 12 bits; the positions above v's bits do not matter)
    auto deposit = [](uint32_t v, uint64_t bits) {
        uint32_t o = 0;
        static_for<12>([&](auto k) { o |= ((v >> k) & 1u) << ((uint32_t)(bits >> (5 * k)) & 31u); });
        return o;
    };
    const uint32_t ob = deposit(tno, a.ob);
    const uint32_t j = ((uint32_t)tid << a.lsplit) | sub;   // this thread's state in the tile
    const uint32_t at = ob | deposit(sub, a.tb) | deposit((uint32_t)tid, a.tbt);
    const bool rd0 = !(a.diag && a.fresh) && a.lz_mode != 1;
    V y{};
    if (rd0) y = v0[at];
    // the whole tile, SPLIT_ROUND states a thread at a time: tid's address, and the bits above the
    // workgroup's size per round
    const int rounds = 1 << a.lsplit;
    const uint32_t a0 = ob | deposit((uint32_t)tid, a.tb);
    Real sr[SPLIT_ROUND], si[SPLIT_ROUND];   // (components: a V[] array is not kept in registers)
    auto fetch = [&](int g) {
        static_for<SPLIT_ROUND>([&](auto I) {
            if (g + I < rounds) {
                const V t = v1[a0 | deposit((uint32_t)(g + I), a.tbh)];
                sr[I] = t.x;
                si[I] = t.y;
            }
        });
    };
    auto stage = [&](int g) {
        static_for<SPLIT_ROUND>([&](auto I) {
            if (g + I < rounds) {
                V t;
                t.x = sr[I];
                t.y = si[I];
                tile[tid + tpb * (g + I)] = t;
            }
        });
    };
    fetch(0);
    const int col = (int)(j & (uint32_t)(a.ncol - 1));
    const A colsc = a.colscale ? (A)a.colscale[col] : (A)1;
    const A ys = (a.diag && a.yscale) ? (A)a.yscale[col] : (A)1;
    double lar = 0.0, lai = 0.0;
    if (a.lz_mode == 2) {
        lar = (double)colsc * a.lz_prd[2 * col];
        lai = (double)colsc * a.lz_prd[2 * col + 1];
    }
    const int dprog = a.diag ? diagp->nprog : 0;
    const uint32_t dpa = dprog ? diagp->prog_a[tid & 63] : 0u;
    const uint32_t dpb = dprog ? diagp->prog_b[tid & 63] : 0u;
    {
        uint32_t w = 0;
#pragma unroll 8
        for (int t = 0; t < a.nterm; ++t) w ^= terms[a.first_term + t].flags;
        asm volatile("" ::"s"(w));
    }
    stage(0);
    for (int g = SPLIT_ROUND; g < rounds; g += SPLIT_ROUND) {
        fetch(g);
        stage(g);
    }
    __syncthreads();
    const V x = tile[j];

    A ar = (A)0, ai = (A)0;
    if (a.diag) {
        const uint32_t st = (uint32_t)(at >> a.colbits);
        double dr, di;
        if (dprog) {   // the lane program (see DiagDev), the whole state at once
            dr = diagp->c0r + a.shift;
            di = diagp->c0i;
            uint32_t cnt = 0u;
            for (int e = 0; e < dprog; ++e) {
                const uint32_t pa = (uint32_t)__builtin_amdgcn_readlane((int)dpa, e);
                const uint32_t m = (uint32_t)__builtin_amdgcn_readlane((int)dpb, e);
                cnt += (uint32_t)__popc(((pa & 64u) ? (st ^ (st >> (pa & 63u))) : st) & m);
                if (pa & 128u) {
                    const int c = (int)((pa >> 8) & 7u);
                    const uint64_t wrb = (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)dpa, 48 + c) |
                                         ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)dpa, 56 + c) << 32);
                    const uint64_t wib = (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)dpb, 48 + c) |
                                         ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)dpb, 56 + c) << 32);
                    dr = fma((double)cnt, __longlong_as_double((long long)wrb), dr);
                    di = fma((double)cnt, __longlong_as_double((long long)wib), di);
                    cnt = 0u;
                }
            }
        } else {
            dr = diag_value_re(*diagp, st, di) + a.shift;
        }
        ar = (A)(dr * (double)x.x - di * (double)x.y);
        ai = (A)(dr * (double)x.y + di * (double)x.x);
    }

    const uint32_t jb = j * (uint32_t)sizeof(V);
    auto run = [&](int t, const int e, auto CXc) {
        constexpr bool CX = decltype(CXc)::value;
        // slot bits are kept whole: flip mask mlo | mhi, selector slo | shi (one thread per slot)
        auto read = [&](const TmTerm &T) {
            return *reinterpret_cast<const V *>(smem_raw + (jb ^ (T.mlo * (uint32_t)sizeof(V))));
        };
        auto add = [&](const TmTerm &T, const V &p) {
            const bool f = (__popc(j & T.slo) + __popc(ob & (uint32_t)T.sout)) & 1;
            const A c0r = (A)uniform(T.c0r), c1r = (A)uniform(T.c1r);
            const A cr = f ? c1r : c0r;
            ar = fma(cr, (A)p.x, ar);
            if constexpr (CX) {
                const A c0i = (A)uniform(T.c0i), c1i = (A)uniform(T.c1i);
                const A ci = f ? c1i : c0i;
                ar = fma(-ci, (A)p.y, ar);
                ai = fma(cr, (A)p.y, ai);
                ai = fma(ci, (A)p.x, ai);
            } else {
                ai = fma(cr, (A)p.y, ai);
            }
        };
        for (; t + 3 < e; t += 4) {
            const TmTerm T0 = terms[t], T1 = terms[t + 1], T2 = terms[t + 2], T3 = terms[t + 3];
            const V p0 = read(T0), p1 = read(T1), p2 = read(T2), p3 = read(T3);
            add(T0, p0);
            add(T1, p1);
            add(T2, p2);
            add(T3, p3);
        }
        for (; t < e; ++t) {
            const TmTerm T0 = terms[t];
            add(T0, read(T0));
        }
    };
    run(a.first_term, a.first_term + a.nreal, std::false_type{});
    run(a.first_term + a.nreal, a.first_term + a.nterm, std::true_type{});

    if (a.colscale) {
        ar *= colsc;
        ai *= colsc;
    }
    double2 *cs = reinterpret_cast<double2 *>(smem_raw + (sizeof(V) << a.K));   // for the partial sums
    if (a.lz_mode == 2) {
        const double wr0 = (double)fma(ys, (A)y.x, ar);
        const double wi0 = (double)fma(ys, (A)y.y, ai);
        const double xr_ = (double)x.x * (double)colsc, xi_ = (double)x.y * (double)colsc;
        // (rounded as hv_s12_tm's expressions are contracted)
        const double wr = wr0 - fma(lar, xr_, -(lai * xi_));
        const double wi = wi0 - fma(lai, xr_, lar * xi_);
        cs[tid] = make_double2(wr, wi);
        ar = (A)fma(-lar, xr_, wr0);
        ai = (A)fma(-lar, xi_, wi0);
    } else {
        cs[tid] = make_double2((double)ar, (double)ai);
        if (rd0) {
            ar = fma(ys, (A)y.x, ar);
            ai = fma(ys, (A)y.y, ai);
        }
    }
    if (a.lz_mode != 1) {
        V o;
        o.x = (Real)ar;
        o.y = (Real)ai;
        v0[at] = o;
    }
    __syncthreads();
    // slot j belongs to thread j mod 256 of the 256: here nv of them, slots nv apart in tid
    const int nv = 256 >> a.lsplit, nr = tpb / nv;
    double2 *red = cs + tpb;
    if (tid < nv) {
        double pr_re = 0.0, pr_im = 0.0;
        for (int r = 0; r < nr; ++r) {
            const double2 c = cs[tid + nv * r];
            if (a.lz_mode == 2) {
                pr_re = fma(c.x, c.x, fma(c.y, c.y, pr_re));
            } else {
                const V z = tile[((uint32_t)(tid + nv * r) << a.lsplit) | sub];
                const double hr = c.x, hi = c.y;
                pr_re += (double)z.x * hr + (double)z.y * hi;
                pr_im += (double)z.x * hi - (double)z.y * hr;
            }
        }
        red[tid] = make_double2(pr_re, pr_im);
    }
    __syncthreads();
    // halvings while the partner is here and of the same column
    const int keep = max(a.ncol >> a.lsplit, 1);
    for (int s = nv / 2; s >= keep; s >>= 1) {
        if (tid < s) {
            red[tid].x += red[tid + s].x;
            red[tid].y += red[tid + s].y;
        }
        __syncthreads();
    }
    if (tid < keep) {   // row tno: [sums still to be halved][column]
        const size_t o = (size_t)tno * max(a.ncol, 1 << a.lsplit) + ((size_t)tid << a.lsplit) + sub;
        partial[2 * o] = red[tid].x;
        partial[2 * o + 1] = red[tid].y;
    }
}

// the sums of hv_s12_split's rows: each row's `width` values are halved down to ncol columns, then the
// rows are added as reduce_partials adds them
__global__ __launch_bounds__(256) void reduce_split(const double *__restrict__ partial, int nrows, int ncol, int width,
                                                    double *__restrict__ out)
{
    __shared__ double red[256];
    const int c = blockIdx.x >> 1, part = blockIdx.x & 1, tid = threadIdx.x;
    double s = 0.0;
    for (int b = tid; b < nrows; b += 256) {
        const double *row = partial + (size_t)b * 2 * width + part;
        double v[16];
        const int m = width / ncol;   // at most 16
#pragma unroll
        for (int i = 0; i < 16; ++i) v[i] = i < m ? row[2 * (c + ncol * i)] : 0.0;
#pragma unroll
        for (int h = 8; h > 0; h >>= 1)
            if (h < m)
#pragma unroll
                for (int i = 0; i < h; ++i) v[i] += v[i + h];
        s += v[0];
    }
    red[tid] = s;
    __syncthreads();
    for (int k = 128; k > 0; k >>= 1) {
        if (tid < k) red[tid] += red[tid + k];
        __syncthreads();
    }
    if (tid == 0) out[blockIdx.x] = red[0];
}

// out[c] = sum over rows of partial[row][c]: one block per column, fixed strides and a
// fixed tree, so the result is the same for the same partials
__global__ __launch_bounds__(256) void reduce_partials(const double *__restrict__ partial, int nrows, int ncol2,
                                                       double *__restrict__ out, int accumulate)
{
    __shared__ double red[256];
    const int c = blockIdx.x, tid = threadIdx.x;
    double s = 0.0;
    for (int b = tid; b < nrows; b += 256) s += partial[(size_t)b * ncol2 + c];
    red[tid] = s;
    __syncthreads();
    for (int k = 128; k > 0; k >>= 1) {
        if (tid < k) red[tid] += red[tid + k];
        __syncthreads();
    }
    if (tid == 0) out[c] = accumulate ? out[c] + red[0] : red[0];
}

int reduce_rows_result(pned_ctx *ctx, int nrows, int ncol2)
{
    hipLaunchKernelGGL(reduce_partials, dim3(ncol2), dim3(256), 0, ctx->stream, ctx->d_partial, nrows, ncol2,
                       ctx->d_result, 0);
    PNED_HIP(hipGetLastError());
    return PNED_OK;
}

template <typename Real, int TPB, int R>
static int launch_pass(pned_ctx *ctx, const void *v1, void *v0, const DiagDev *ddiag, const PassDev *pd,
                       const PassArgs &a, double *partial, int grid)
{
    using V = typename C2<Real>::T;
    size_t lds = sizeof(V) * (size_t)TPB * R;
    size_t need_red = sizeof(double) * 2 * TPB;
    if (lds < need_red) lds = need_red;
    auto kern = hv_s12_pass<Real, TPB, R>;
    PNED_HIP(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(kern, dim3(grid), dim3(TPB), lds, ctx->stream, (const V *)v1, (V *)v0,
                       ctx->d_terms, ddiag, pd, a, partial);
    PNED_HIP(hipGetLastError());
    return PNED_OK;
}

// the instances of dispatch_pass
static bool has_pass(int TPB, int R)
{
    if (TPB == 256 || TPB == 512) return R <= 32 && R > TPB / 512;
    return R == 1 && (TPB == 128 || TPB == 64 || TPB == 32 || TPB == 16);
}

template <typename Real>
static int dispatch_pass(pned_ctx *ctx, int TPB, int R, const void *v1, void *v0,
                         const DiagDev *ddiag, const PassDev *pd, const PassArgs &a, double *partial, int grid)
{
#define PNED_CASE(T_, R_) \
    if (TPB == T_ && R == R_) return launch_pass<Real, T_, R_>(ctx, v1, v0, ddiag, pd, a, partial, grid);
    PNED_CASE(256, 32) PNED_CASE(256, 16) PNED_CASE(256, 8) PNED_CASE(256, 4) PNED_CASE(256, 2)
    PNED_CASE(256, 1) PNED_CASE(128, 1) PNED_CASE(64, 1) PNED_CASE(32, 1) PNED_CASE(16, 1)
    PNED_CASE(512, 32) PNED_CASE(512, 16) PNED_CASE(512, 8) PNED_CASE(512, 4) PNED_CASE(512, 2)
#undef PNED_CASE
    return fail(PNED_E_UNSUPPORTED, "no H.v kernel instance for this tile shape");
}

// LDS the term-major kernel stages per-column coefficients in (batch contexts)
static size_t tm_coef_bytes(int nop, int nterm, bool diag, size_t ngroups)
{
    if (nop <= 1) return 0;
    return sizeof(double) * ((size_t)4 * nterm * nop + (diag ? (size_t)2 * (ngroups + 1) * nop : 0));
}
static size_t tm_coef_bytes(const PassArgs &a) { return tm_coef_bytes(a.nop, a.nterm, a.diag != 0, a.ngroups); }
// a pass's tile and coefficients
static size_t tm_lds(const S12Plan &pl, const PassPlan &pp, bool c128)
{
    return ((size_t)(c128 ? 16 : 8) << pp.K) + tm_coef_bytes(pl.nop, pp.nterm, pp.diag, pl.diag.size());
}
constexpr size_t LDS_LIMIT = 160 * 1024;

bool s12_tm_fits(const S12Plan &pl, int dtype)
{
    for (const PassPlan &pp : pl.passes)
        if (tm_lds(pl, pp, dtype == PNED_C128) > LDS_LIMIT) return false;
    return true;
}
// a batched tile of a single-operator context holds the columns of one 256-byte run (32
// complex64 or 16 complex128 values per state); more columns run in groups
constexpr size_t COL_GROUP_BYTES = 256;

template <typename Real, int TPB, int R, int S>
static int launch_tm(pned_ctx *ctx, const void *v1, void *v0, const TmTerm *tm, const DiagDev *ddiag,
                     const PassDev *pd, const PassArgs &a, double *partial, int grid)
{
    using V = typename C2<Real>::T;
    size_t lds = sizeof(V) * (size_t)TPB * R + tm_coef_bytes(a);
    size_t need_red = sizeof(double) * 2 * TPB;
    if (lds < need_red) lds = need_red;
    auto kern = hv_s12_tm<Real, TPB, R, S>;
    PNED_HIP(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(kern, dim3(grid), dim3(TPB), lds, ctx->stream, (const V *)v1, (V *)v0, tm, ddiag, pd, a,
                       partial);
    PNED_HIP(hipGetLastError());
    return PNED_OK;
}

// term-major instances: the prefetched v1 of R slots plus the accumulators and v0 of one
// sweep of S slots stay in registers; S is chosen so that nothing spills at the block's
// occupancy (1024 threads leave 128 registers per lane, 512 threads 256)
template <typename Real>
static bool has_tm(int TPB, int R)
{
    if (TPB != 256 && TPB != 512 && TPB != 1024) return false;
    if (sizeof(Real) == 8) return R == 1 || R == 2 || R == 4 || R == 8 || (R == 16 && TPB <= 512);
    return R == 1 || R == 2 || R == 4 || R == 8 || R == 16 || (R == 32 && TPB <= 512);
}

template <typename Real>
static int dispatch_tm(pned_ctx *ctx, int TPB, int R, const void *v1, void *v0, const TmTerm *tm,
                       const DiagDev *ddiag, const PassDev *pd, const PassArgs &a, double *partial, int grid)
{
#define PNED_CASE(T_, R_, S_) \
    if (TPB == T_ && R == R_) return launch_tm<Real, T_, R_, S_>(ctx, v1, v0, tm, ddiag, pd, a, partial, grid);
    if constexpr (sizeof(Real) == 8) {
        PNED_CASE(256, 16, 8) PNED_CASE(256, 8, 8) PNED_CASE(256, 4, 4) PNED_CASE(256, 2, 2) PNED_CASE(256, 1, 1)
        PNED_CASE(512, 16, 8) PNED_CASE(512, 8, 4) PNED_CASE(512, 4, 4) PNED_CASE(512, 2, 2) PNED_CASE(512, 1, 1)
        PNED_CASE(1024, 8, 4) PNED_CASE(1024, 4, 4) PNED_CASE(1024, 2, 2) PNED_CASE(1024, 1, 1)
    } else {
        PNED_CASE(256, 32, 16) PNED_CASE(256, 16, 16) PNED_CASE(256, 8, 8) PNED_CASE(256, 4, 4)
        PNED_CASE(256, 2, 2) PNED_CASE(256, 1, 1)
        PNED_CASE(512, 32, 16) PNED_CASE(512, 16, 16) PNED_CASE(512, 8, 8) PNED_CASE(512, 4, 4)
        PNED_CASE(512, 2, 2) PNED_CASE(512, 1, 1)
        PNED_CASE(1024, 16, 8) PNED_CASE(1024, 8, 8) PNED_CASE(1024, 4, 4) PNED_CASE(1024, 2, 2)
        PNED_CASE(1024, 1, 1)
    }
#undef PNED_CASE
    return fail(PNED_E_UNSUPPORTED, "no term-major H.v kernel instance for this tile shape");
}

template <typename Real>
static int launch_split(pned_ctx *ctx, const void *v1, void *v0, const TmTerm *tm, const SmallArgs &a, double *partial,
                        int tiles)
{
    using V = typename C2<Real>::T;
    const int tpb = 1 << (a.K - a.lsplit);
    const size_t lds = (sizeof(V) << a.K) + sizeof(double2) * ((size_t)tpb + 256);
    auto kern = hv_s12_split<Real>;
    PNED_HIP(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(kern, dim3(tiles << a.lsplit), dim3(tpb), lds, ctx->stream, (const V *)v1, (V *)v0, tm,
                       ctx->d_diag, a, partial);
    PNED_HIP(hipGetLastError());
    return PNED_OK;
}

// log2 of hv_s12_split's workgroups per tile, or -1 where a plan stays with hv_s12_tm.  An untuned plan of
// one operator, tiles of 2^8 .. 2^12 states (2^13 complex64 ones).  Above a number of elements staging a
// tile several times costs more than the chain (us per H.v, split kernel against whole tiles):
// - complex64, or more than 16 complex128 columns, 2^17: 2^18 complex64 elements 49.6 against 47; 2^17 as
//   10 sites with 128 columns, whose tiles hold few sites and run in many passes, 133 against 141
// - 2 to 16 complex128 columns 2^16: 14 sites with 8 columns 36.0 against 32.4, 16 with 2 44.9 against 39.1
// - one complex128 column 2^17, or 2^18 where the passes have 16 terms or more on average: 18 sites in two
//   passes, with field (22 a pass) 62 against 68 on 256 threads, without (13) 56.8 against 54.9, and 43 on
//   the 1024 threads such a plan takes.  (1024 threads are faster with field as well, 50, but not with the
//   sums of 256 threads bit for bit.)
// Workgroups of 1024 threads where that makes 256 or more of them, else smaller ones, down to 256 threads
static int split_plan(const pned_ctx *ctx, const S12Plan &pl, int colbits, bool c128)
{
    if (ctx->s12_kernel != 1 || pl.nop > 1 || ctx->tune_threads > 0 || ctx->tune_tile_bits > 0) return -1;
    if (colbits > 8) return -1;   // its sums follow those of 256 threads, one column each at most
    const bool many = pl.devterms.size() >= 16 * pl.passes.size();
    if (ctx->n + colbits > (!c128 || colbits > 4 ? 17 : colbits > 0 ? 16 : many ? 18 : 17) || pl.passes.empty()) return -1;
    const int K = pl.passes[0].K;
    for (const PassPlan &pp : pl.passes)
        if (pp.K != K || K < 8 || K > (c128 ? 12 : 13) || pp.ob.size() > 10) return -1;
    int ls = std::max(0, K - 10);
    const int tiles = (int)pl.passes[0].ob.size();
    while (tiles + ls < 8 && ls < 4 && K - ls > 8) ++ls;
    return ls;
}

// Tile-coordinate term table of one pass (see TmTerm), sorted into the term-major
// kernel's categories: 0 real, 1 real with register selector bits, 2 complex, 3 complex
// with register selector bits (batch contexts: every term complex).  ncat gets the counts.
// The order in which a state sums its terms is a function of the plan and of order_tpb alone,
// whatever the thread count: the categories sort by the register bits that order_tpb threads
// would leave (the looser loop of 1 and 3 is right for every selector; where TPB leaves more
// register bits than order_tpb, all real or complex terms take it).
// colbits: the plan's column bits; outer selector bits at or above them sit gap bits higher
// in memory (column groups)
static void build_tm_terms(const S12Plan &pl, const PassPlan &pp, int TPB, int order_tpb, int colbits, int gap,
                           std::vector<TmTerm> &out, int ncat[4])
{
    const int LT = __builtin_ctz(TPB), LO = __builtin_ctz(order_tpb);
    uint64_t tilemask = 0;
    for (int b : pp.tb) tilemask |= 1ull << b;
    std::vector<TmTerm> cat[4];
    for (int i = 0; i < pp.nterm; ++i) {
        const DevTerm &d = pl.devterms[pp.first_term + i];
        TmTerm t{};
        t.mlo = d.tmask & (uint32_t)(TPB - 1);
        t.mhi = d.tmask >> LT;
        const uint64_t selm = (uint64_t)d.selmask << colbits;
        uint32_t stile = 0;
        for (int k = 0; k < pp.K; ++k)
            if (selm >> pp.tb[k] & 1) stile |= 1u << k;
        t.slo = stile & (uint32_t)(TPB - 1);
        t.shi = stile >> LT;
        const uint64_t so = selm & ~tilemask;
        t.sout = (so & ((1ull << colbits) - 1)) | ((so >> colbits) << (colbits + gap));
        const bool cx = !d.is_real || pl.nop > 1;
        t.flags = (cx ? 1u : 0u) | ((t.shi != 0) ? 2u : 0u);
        t.term = (uint32_t)(pp.first_term + i);
        t.c0r = d.c0r;
        t.c0i = d.c0i;
        t.c1r = d.c1r;
        t.c1i = d.c1i;
        cat[(cx ? 2 : 0) + ((stile >> LO) != 0 ? 1 : 0)].push_back(t);
    }
    for (int c = 0; c < 4; ++c) {
        ncat[c] = (int)cat[c].size();
        out.insert(out.end(), cat[c].begin(), cat[c].end());
    }
    for (int c = 0; c < 4; c += 2)
        for (const TmTerm &t : cat[c])
            if (t.shi != 0) {
                ncat[c + 1] += ncat[c];
                ncat[c] = 0;
                break;
            }
}

// ------------------------------------------------------------------------------------
// Scratch of the allocation-free H.v (pned_p_mltply_v3_noalloc): the per-block partial
// sums of <v1|H|v1> of every pass.  One array per GPU for the life of the process; its
// device address is looked up once per device when the first context on that device is
// created, and host code only ever passes that address (the array's name is a host-side
// stand-in).  Calls on one GPU share it, so overlapping calls on one GPU race.
// ------------------------------------------------------------------------------------
constexpr size_t NOALLOC_SCRATCH_DOUBLES = PNED_NOALLOC_SCRATCH_BYTES / sizeof(double);
static __device__ __align__(256) double scratch[NOALLOC_SCRATCH_DOUBLES];
constexpr int NOALLOC_MAX_DEVICES = 64;
static std::mutex g_scratch_mu;
static double *g_scratch_ptr[NOALLOC_MAX_DEVICES];

int noalloc_scratch_init(int device)
{
    if (device < 0 || device >= NOALLOC_MAX_DEVICES) return fail(PNED_E_ARG, "device index out of range");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch_ptr[device]) return PNED_OK;
    int cur = 0;
    PNED_HIP(hipGetDevice(&cur));
    if (cur != device) PNED_HIP(hipSetDevice(device));
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (cur != device) PNED_HIP(hipSetDevice(cur));
    if (e != hipSuccess || p == nullptr)
        return fail(PNED_E_HIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
    g_scratch_ptr[device] = static_cast<double *>(p);
    return PNED_OK;
}

static double *noalloc_scratch(int device)
{
    if (device < 0 || device >= NOALLOC_MAX_DEVICES) return nullptr;
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    return g_scratch_ptr[device];
}

// Infinity Cache, shared by the XCDs
constexpr size_t CACHE_BYTES = (size_t)256 << 20;

// consecutive low bits of an ascending bit list: runs of 2^n elements are contiguous
static int contiguous_bits(const std::vector<int> &b)
{
    int n = 0;
    while (n < (int)b.size() && b[n] == n) ++n;
    return n;
}

// (see hv_s12_tm) whole 128-byte lines in every pass: one pass with runs of 64 bytes reads each line
// twice (24 sites with 8 complex64 columns and a field, where the first pass alone has longer runs: 4.75 ms
// per H.v, 3.86 without the hint)
int s12_nt_streams(const S12Plan &pl, int dtype, size_t vec_bytes)
{
    int run = 31;
    for (const PassPlan &pp : pl.passes) run = std::min(run, contiguous_bits(pp.tb));
    if (2 * vec_bytes <= CACHE_BYTES || ((size_t)(dtype == PNED_C128 ? 16 : 8) << run) < 128) return 0;
    return vec_bytes > CACHE_BYTES ? NT_V1 | NT_V0 : NT_V0;
}

// Threads of the untuned term-major plan, by its tile size (complex128 figures: one column with
// field, us per H.v).  2^12-state tiles 1024 threads up to 2^21 elements (N=20 57.9, on 512 68), 512
// above (N=24 533 against 565: two blocks per CU), but 1024 with columns of one operator (N=20 with
// 8 columns 277 against 344); one operator per column 512 above as well (5 batch steps, N=20 with 8
// columns 2.41 ms against 2.52) while two of its blocks fit a CU (20 sites with 64 operators, up to 98 KB a
// block: 5.39 ms per H.v on 512, 4.60 on 1024).  2^11-state tiles 512: 4 slots a thread, 105 VGPRs against 169 on
// 256 threads (5 batch steps, N=16 with 8 columns 464 us against 528, N=18 with 2 446 against 497;
// 1024 threads 1000 against 897 at N=18 with 8).  2^13 1024 (N=28 9.08 ms, on 512 13.9).  complex64:
// 2^12 512 (N=24 383, on 1024 472), 2^13 1024 (N=28 5.8 ms), 2^14 512 (1024 spill; N=24 with 64 columns
// 28.7 against 31.7 ms).
static int default_threads(const pned_ctx *ctx, const S12Plan &pl, int colbits, bool c128)
{
    const int K = pl.passes.empty() ? 12 : pl.passes[0].K;
    const bool big = (double)ctx->dim * (double)(1ull << colbits) > (double)(1ull << 21);
    if (K <= 10) return 256;
    if (K == 11) return 512;
    if (!c128) return K == 13 ? 1024 : 512;
    bool two = K == 12 && big && (colbits == 0 || pl.nop > 1);
    for (const PassPlan &pp : pl.passes) two = two && tm_lds(pl, pp, c128) <= LDS_LIMIT / 2;
    return two ? 512 : 1024;
}

// the thread count whose register slots order a pass's terms (see build_tm_terms)
static int order_threads(const pned_ctx *ctx, int colbits)
{
    return (double)ctx->dim * (double)(1ull << colbits) > (double)(1ull << 25) ? 1024 : 256;
}

// noalloc: the caller's plan, pass tables and buffers must already exist; partials go to
// part_ext (cap doubles) and the sums of <v1|H|v1> to result_ext (device memory).  Nothing
// is allocated and the stream is not synchronised.
static int hv_s12_run(pned_ctx *ctx, const pned_vec *v1, pned_vec *v0, double eperbd, bool fresh,
                      double *prdct_host, const double *d_colscale, const double *d_yscale, bool *lz_fused,
                      bool noalloc, double *part_ext, size_t part_cap, double *result_ext);

int launch_hv_s12(pned_ctx *ctx, const pned_vec *v1, pned_vec *v0, double eperbd, bool fresh,
                  double *prdct_host, const double *d_colscale, const double *d_yscale, bool *lz_fused)
{
    return hv_s12_run(ctx, v1, v0, eperbd, fresh, prdct_host, d_colscale, d_yscale, lz_fused, false, nullptr, 0,
                      nullptr);
}

static int hv_s12_run(pned_ctx *ctx, const pned_vec *v1, pned_vec *v0, double eperbd, bool fresh,
                      double *prdct_host, const double *d_colscale, const double *d_yscale, bool *lz_fused,
                      bool noalloc, double *part_ext, size_t part_cap, double *result_ext)
{
    if (lz_fused) *lz_fused = false;
    const int nvec = v1->nvec;
    int colbits = 0;
    while ((1 << colbits) < nvec) ++colbits;
    if ((1 << colbits) != nvec)
        return fail(PNED_E_UNSUPPORTED, "batched H.v needs a power-of-two column count");
    // A single-operator batch wider than one 256-byte run of columns runs in column groups: the
    // plan's tiles hold that run's column bits, the higher column bits are fixed per launch
    // (one launch per group and pass, base pointers moved by the group), so a tile spends its
    // other bits on sites and a pass covers more terms (N=24 with 64 columns: 4 -> 3 passes).
    // Plan positions at or above cg move up by gap bits in memory (expand).
    // Groups are taken only where they save a pass (ensure_s12_plan_cols).
    const int run_bits = __builtin_ctzll(COL_GROUP_BYTES / (v1->dtype == PNED_C128 ? 16 : 8));
    int cg = colbits;
    if (noalloc) {
        if (ctx->plan_req_colbits != colbits || ctx->plan_colbits < 0 || ctx->plan_dtype != v1->dtype ||
            ctx->pd_dev == nullptr || ctx->pd_gap != colbits - ctx->plan_colbits)
            return fail(PNED_E_ARG, "no H.v plan for this vector shape yet: call pned_p_mltply_v3 once with "
                                    "vectors of this shape first (that call allocates the plan's tables)");
        cg = ctx->plan_colbits;
    } else {
        PNED_TRY(ensure_s12_plan_cols(ctx, colbits, run_bits, v1->dtype, &cg));
    }
    const int gap = colbits - cg, ngrp = 1 << gap, ncol_t = 1 << cg;
    auto expand = [cg, gap](int b) { return b < cg ? b : b + gap; };
    const S12Plan &pl = ctx->s12;
    if (pl.nop > 1 && pl.nop != nvec)
        return fail(PNED_E_ARG, "a batch context's vectors need one column per operator");
    const int npass = (int)pl.passes.size();
    const int grid_cap = 4096;
    // partial layout: [pass][block][2*ncol] (plus one pass for a fused Lanczos step)
    if (noalloc) {
        const size_t need = (size_t)npass * grid_cap * 2 * nvec;
        if (need > part_cap)
            return fail(PNED_E_ARG, "allocation-free H.v: " + std::to_string(npass) + " passes x " +
                                        std::to_string(nvec) + " columns need " + std::to_string(need * 8) +
                                        " bytes of partial sums, more than the " +
                                        std::to_string(part_cap * 8) + "-byte static scratch");
    } else {
        size_t need = (size_t)(npass + 1) * grid_cap * 2 * nvec + 64;
        PNED_TRY(ensure_partial(ctx, need));
        PNED_TRY(ensure_result(ctx, 4 * (size_t)nvec + 8));
    }
    double *const part_base = noalloc ? part_ext : ctx->d_partial;
    const bool c128 = v1->dtype == PNED_C128;
    const size_t esz = c128 ? 16 : 8;
    // per-pass address tables (rebuilt when the plan or the thread count changes)
    const int lsplit = split_plan(ctx, pl, colbits, c128);
    const bool small = lsplit >= 0;
    // (hv_s12_split keeps a slot's bits whole, as a table for 2^13 threads would)
    const int TPBpref = small ? 8192 : (ctx->tune_threads == 256 || ctx->tune_threads == 512 || ctx->tune_threads == 1024)
                            ? ctx->tune_threads
                            : (ctx->s12_kernel == 1 ? default_threads(ctx, pl, colbits, c128) : 512);
    std::vector<int> tpb(npass), rr(npass), tmk(npass);   // tmk: the pass takes the term-major kernel
    for (int p = 0; p < npass; ++p) {
        const PassPlan &pp = pl.passes[p];
        int T = TPBpref;
        while (T > 16 && T > (1 << pp.K)) T >>= 1;
        tmk[p] = ctx->s12_kernel == 1 && !small &&
                 (c128 ? has_tm<double>(T, (1 << pp.K) / T) : has_tm<float>(T, (1 << pp.K) / T)) &&
                 tm_lds(pl, pp, c128) <= LDS_LIMIT;
        // a default thread count is the term-major kernel's; a pass that leaves it (coefficients beyond
        // the LDS) runs the state-major kernel on 256 threads, 512 for 2^14 states
        if (ctx->s12_kernel == 1 && !small && !tmk[p] && ctx->tune_threads == 0)
            T = std::min(T, pp.K > 13 ? 512 : 256);
        tpb[p] = T;
        rr[p] = (1 << pp.K) / T;
        if (rr[p] > PD_HI) return fail(PNED_E_UNSUPPORTED, "tile too large for the thread count");
        if ((int)pp.ob.size() > 22) return fail(PNED_E_UNSUPPORTED, "too many outer bits");
        // (before the first launch: v0 is not touched by a call that fails)
        if (!small && !tmk[p] && !has_pass(T, rr[p]))
            return fail(PNED_E_UNSUPPORTED, "no H.v kernel instance for this tile shape");
    }
    if (noalloc && (ctx->pd_threads != TPBpref || ctx->pd_tpb != tpb))
        return fail(PNED_E_ARG, "no H.v plan for this thread count yet: call pned_p_mltply_v3 once after "
                                "changing the tuning (that call rebuilds the plan's tables)");
    if (ctx->pd_threads != TPBpref || ctx->pd_tpb != tpb || ctx->pd_gap != gap || ctx->pd_dev == nullptr) {
        std::vector<PassDev> host(npass);
        for (int p = 0; p < npass; ++p) {
            const PassPlan &pp = pl.passes[p];
            PassDev &d = host[p];
            std::memset(&d, 0, sizeof(PassDev));
            if (small) continue;   // (no address tables)
            const int LT = __builtin_ctz(tpb[p]);
            for (int t = 0; t < tpb[p]; ++t) {
                uint64_t o = 0;
                for (int k = 0; k < LT; ++k)
                    if ((t >> k) & 1) o |= 1ull << expand(pp.tb[k]);
                d.lo[t] = o;
            }
            for (int r = 0; r < rr[p]; ++r) {
                uint64_t o = 0;
                for (int k = 0; LT + k < pp.K; ++k)
                    if ((r >> k) & 1) o |= 1ull << expand(pp.tb[LT + k]);
                d.hi[r] = o;
            }
            const int no = (int)pp.ob.size(), nlo = no < 11 ? no : 11, nhi = no - nlo;
            for (int x = 0; x < (1 << nlo); ++x) {
                uint64_t o = 0;
                for (int k = 0; k < nlo; ++k)
                    if ((x >> k) & 1) o |= 1ull << expand(pp.ob[k]);
                d.blo[x] = o;
            }
            for (int x = 0; x < (1 << nhi); ++x) {
                uint64_t o = 0;
                for (int k = 0; k < nhi; ++k)
                    if ((x >> k) & 1) o |= 1ull << expand(pp.ob[nlo + k]);
                d.bhi[x] = o;
            }
        }
        std::vector<TmTerm> tmh;
        ctx->tm_ncat.assign(4 * (size_t)npass, 0);
        for (int p = 0; p < npass; ++p) {
            int T = ctx->tune_threads > 0 ? TPBpref : order_threads(ctx, colbits);
            while (T > 16 && T > (1 << pl.passes[p].K)) T >>= 1;
            build_tm_terms(pl, pl.passes[p], tpb[p], T, cg, gap, tmh, &ctx->tm_ncat[4 * p]);
        }
        if (tmh.empty()) tmh.push_back(TmTerm{});
        PNED_HIP(hipStreamSynchronize(ctx->stream));
        if (ctx->pd_dev) PNED_HIP(hipFree(ctx->pd_dev));
        ctx->pd_dev = nullptr;
        if (ctx->d_tm) PNED_HIP(hipFree(ctx->d_tm));
        ctx->d_tm = nullptr;
        PNED_HIP(hipMalloc(&ctx->pd_dev, sizeof(PassDev) * npass));
        PNED_HIP(hipMemcpy(ctx->pd_dev, host.data(), sizeof(PassDev) * npass, hipMemcpyHostToDevice));
        PNED_HIP(hipMalloc((void **)&ctx->d_tm, sizeof(TmTerm) * tmh.size()));
        PNED_HIP(hipMemcpy(ctx->d_tm, tmh.data(), sizeof(TmTerm) * tmh.size(), hipMemcpyHostToDevice));
        // the diagonal pass's lane program split by that pass's register bits
        if (ctx->d_diag_tm) PNED_HIP(hipFree(ctx->d_diag_tm));
        ctx->d_diag_tm = nullptr;
        for (int p = 0; p < npass && !small && pl.nop <= 1 && ctx->diag_host.nprog > 0; ++p) {
            const PassPlan &pp = pl.passes[p];
            if (!pp.diag) continue;
            uint32_t slot_bits = 0;
            for (int k = __builtin_ctz(tpb[p]); k < pp.K; ++k) slot_bits |= 1u << (pp.tb[k] - cg);
            DiagDev dt;
            if (split_diag_slots(ctx->diag_host, slot_bits, dt)) {
                PNED_HIP(hipMalloc((void **)&ctx->d_diag_tm, sizeof(DiagDev)));
                PNED_HIP(hipMemcpy(ctx->d_diag_tm, &dt, sizeof(DiagDev), hipMemcpyHostToDevice));
            }
        }
        ctx->pd_threads = TPBpref;
        ctx->pd_tpb = tpb;
        ctx->pd_gap = gap;
    }
    // blocks per pass: at least 8 contiguous tiles each (so a block's next-tile loads overlap
    // its terms for most of its tiles) while that leaves one block per CU or more (two where
    // two fit a CU), at most grid_cap.  At N=24 (2048 tiles of 2^13) 256 blocks ran 0.524 ms per
    // H.v against 0.532 with 1024 and 0.554 with 2048; at N=32 4096 blocks of 128 tiles beat 1024
    // and 256 by about 0.5 ms
    auto pass_grid = [&](int p) {
        const uint64_t tc = 1ull << pl.passes[p].ob.size();
        if (small) return (int)tc;   // at most 2^10, times 2^lsplit <= 4 or 16 workgroups
        const uint64_t fill = (tpb[p] <= 512 && tm_lds(pl, pl.passes[p], c128) <= LDS_LIMIT / 2) ? 512 : 256;
        const uint64_t want = std::max<uint64_t>(fill, tc / 8);
        return (int)std::min<uint64_t>(std::min<uint64_t>(tc, want), (uint64_t)grid_cap);
    };
    // partial rows: per column group [pass][block] of 2 ncol_t values, the groups one after another
    int rows_grp = 0;
    for (int p = 0; p < npass; ++p) rows_grp += pass_grid(p);
    // values per partial row and column part, and the sum over rows
    const int width = small ? std::max(ncol_t, 1 << lsplit) : ncol_t;
    auto reduce_rows_of = [&](const double *part, int rows, double *out) -> int {
        if (small)
            hipLaunchKernelGGL(reduce_split, dim3(2 * ncol_t), dim3(256), 0, ctx->stream, part, rows, ncol_t, width, out);
        else
            hipLaunchKernelGGL(reduce_partials, dim3(2 * ncol_t), dim3(256), 0, ctx->stream, part, rows, 2 * ncol_t, out,
                               0);
        PNED_HIP(hipGetLastError());
        return PNED_OK;
    };
    const int nt = s12_nt_streams(pl, v1->dtype, esz * (size_t)ctx->dim * (size_t)nvec);
    int total_rows = 0;
    for (int p = 0; p < npass; ++p) {
        const PassPlan &pp = pl.passes[p];
        PassArgs a{};
        a.K = pp.K;
        a.nouter = (int)pp.ob.size();
        a.tile_count = 1ull << a.nouter;
        a.nlo = a.nouter < 11 ? a.nouter : 11;
        a.colbits = colbits;
        a.first_term = pp.first_term;
        a.nterm = pp.nterm;
        a.diag = pp.diag ? 1 : 0;
        a.fresh = fresh ? 1 : 0;
        a.ncol = ncol_t;
        a.shift = -(double)ctx->ibond * eperbd;
        a.nop = pl.nop;
        a.colcoef = ctx->d_colcoef;
        a.coldiag = ctx->d_coldiag;
        a.colscale = d_colscale;
        a.yscale = d_yscale;
        for (int c = 0; c < 4; ++c) a.ncat[c] = ctx->tm_ncat[4 * p + c];
        a.ngroups = ctx->diag_host.ngroups;
        a.nt = nt;
        const int TPB = tpb[p], R = rr[p];
        const int grid = pass_grid(p);
        const PassDev *pdp = reinterpret_cast<const PassDev *>(ctx->pd_dev) + p;
        SmallArgs sm{};
        if (small) {
            sm.colbits = colbits;
            sm.ncol = ncol_t;
            sm.first_term = a.first_term;
            sm.nreal = a.ncat[0] + a.ncat[1];
            sm.nterm = a.nterm;
            sm.diag = a.diag;
            sm.fresh = a.fresh;
            sm.K = pp.K;
            sm.lsplit = lsplit;
            sm.shift = a.shift;
            auto from = [&](int k0) {   // twelve positions are more than deposit() is ever given bits for
                uint64_t w = 0;
                for (int k = k0; k < pp.K && k < k0 + 12; ++k) w |= (uint64_t)expand(pp.tb[k]) << (5 * (k - k0));
                return w;
            };
            sm.tb = from(0);
            sm.tbt = from(lsplit);
            sm.tbh = from(pp.K - lsplit);
            for (int k = 0; k < a.nouter; ++k) sm.ob |= (uint64_t)expand(pp.ob[k]) << (5 * k);
        }
        const bool tm = tmk[p] != 0;
        const DiagDev *dgp = (pp.diag && ctx->d_diag_tm) ? ctx->d_diag_tm : ctx->d_diag;
        if (!noalloc && lz_fused && p == npass - 1 && p > 0 && (tm || small) && c128 && nvec == 1 && pl.nop <= 1) {
            // deferred-normalisation Lanczos step: this pass's <v1|H v1> share first (no v0
            // traffic), alpha from all passes on the device, then the pass itself forms
            // v0 - Re(alpha) s v1 and the partials of beta^2
            double *part = part_base + (size_t)total_rows * 2 * width;
            auto pass = [&](int mode) -> int {
                a.lz_mode = sm.lz_mode = mode;
                sm.lz_prd = a.lz_prd;
                sm.colscale = a.colscale;
                sm.yscale = a.yscale;
                if (small) return launch_split<double>(ctx, v1->data, v0->data, ctx->d_tm, sm, part, grid);
                return dispatch_tm<double>(ctx, TPB, R, v1->data, v0->data, ctx->d_tm, dgp, pdp, a, part, grid);
            };
            PNED_TRY(pass(1));
            total_rows += grid;
            PNED_TRY(reduce_rows_of(ctx->d_partial, total_rows, ctx->d_result));
            a.lz_prd = ctx->d_result;
            part = ctx->d_partial + (size_t)total_rows * 2 * width;
            PNED_TRY(pass(2));
            PNED_TRY(reduce_rows_of(part, grid, ctx->d_result + 2 * nvec));
            *lz_fused = true;
            return PNED_OK;
        }
        for (int g = 0; g < ngrp; ++g) {
            // column group g: columns g*ncol_t .. (g+1)*ncol_t-1 of every state
            const size_t eo = (size_t)g * ncol_t * esz;
            const void *x = static_cast<const char *>(v1->data) + eo;
            void *y = static_cast<char *>(v0->data) + eo;
            a.colscale = d_colscale ? d_colscale + (size_t)g * ncol_t : nullptr;
            a.yscale = d_yscale ? d_yscale + (size_t)g * ncol_t : nullptr;
            double *part = part_base + ((size_t)g * rows_grp + total_rows) * 2 * width;
            int rc;
            if (small) {
                sm.colscale = a.colscale;
                sm.yscale = a.yscale;
                if (c128)
                    rc = launch_split<double>(ctx, x, y, ctx->d_tm, sm, part, grid);
                else
                    rc = launch_split<float>(ctx, x, y, ctx->d_tm, sm, part, grid);
            } else if (tm) {
                // the term table is in pass order, so the kernel indexes it by first_term as well
                if (c128)
                    rc = dispatch_tm<double>(ctx, TPB, R, x, y, ctx->d_tm, dgp, pdp, a, part, grid);
                else
                    rc = dispatch_tm<float>(ctx, TPB, R, x, y, ctx->d_tm, dgp, pdp, a, part, grid);
            } else if (c128) {
                rc = dispatch_pass<double>(ctx, TPB, R, x, y, ctx->d_diag, pdp, a, part, grid);
            } else {
                rc = dispatch_pass<float>(ctx, TPB, R, x, y, ctx->d_diag, pdp, a, part, grid);
            }
            if (rc != PNED_OK) return rc;
        }
        total_rows += grid;
    }
    const int ncol2 = 2 * nvec;
    double *const out = noalloc ? result_ext : ctx->d_result;
    for (int g = 0; g < ngrp; ++g)
        PNED_TRY(reduce_rows_of(part_base + (size_t)g * rows_grp * 2 * width, rows_grp, out + (size_t)g * 2 * ncol_t));
    if (noalloc) return PNED_OK;
    if (prdct_host) {
        PNED_HIP(hipMemcpyAsync(ctx->h_result, ctx->d_result, sizeof(double) * ncol2,
                                hipMemcpyDeviceToHost, ctx->stream));
        PNED_HIP(hipStreamSynchronize(ctx->stream));
        for (int c = 0; c < ncol2; ++c) prdct_host[c] = ctx->h_result[c];
    }
    return PNED_OK;
}

}  // namespace pned

extern "C" int pned_p_mltply_v3_noalloc(pned_ctx *ctx, const pned_vec *v1, pned_vec *v0, double eperbd,
                                        double *prdct_dev)
{
    using namespace pned;
    PNED_TRY(check_hv_pair(ctx, v1, v0));
    if (!prdct_dev) return fail(PNED_E_ARG, "null prdct_dev");
    if (ctx->q != 2 || ctx->sector_k >= 0)
        return fail(PNED_E_UNSUPPORTED, "the allocation-free H.v covers S=1/2 full-space contexts only");
    double *part = noalloc_scratch(ctx->device);
    if (!part) return fail(PNED_E_HIP, "allocation-free H.v: no scratch address for this device");
    PNED_HIP(hipSetDevice(ctx->device));
    return hv_s12_run(ctx, v1, v0, eperbd, false, nullptr, nullptr, nullptr, nullptr, true, part,
                      NOALLOC_SCRATCH_DOUBLES, prdct_dev);
}
