// hv_sector.hip -- S=1/2 H.v in a fixed-S^z sector basis (the reference's parity_type = 0).
//
// Basis (mk_list12, S_one_half/Hybrid_TPS_parallel.f90:452-578, at one process): the
// states with k set bits in increasing order.  A state's index comes from its two halves
// (right half: the low ihf = (N+1)/2 bits, left half: the rest):
//     index(s) = rank(s & right) + offset(s >> ihf)
// where rank is the position of the right half among right halves of the same popcount
// and offset counts the sector states of every smaller left half -- the reference's
// list3(1,.) - 1 and list3(2,.).  list1 (index -> state) is kept in device memory.
//
// H.v reuses the S=1/2 term decomposition: the diagonal groups act on the state, and a
// two-bit flip term keeps the state in the sector exactly when the two bits differ; the
// context checks at set-up that every other term vanishes (the operator conserves S^z).
// One thread per output index gathers its partners through the two half tables.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "internal.h"

namespace pned {

struct SectorTerm {
    uint32_t mask;       // the two flipped bits
    uint32_t selmask;
    double c0r, c0i, c1r, c1i;
};

__device__ __forceinline__ double sector_diag(const DiagDev &d, uint32_t s, double &im)
{
    double re = d.c0r;
    im = d.c0i;
    for (int g = 0; g < d.ngroups; ++g) {
        const uint32_t f = (d.kind[g] == 0) ? (s & d.mask[g]) : ((s ^ (s >> d.shift[g])) & d.mask[g]);
        const double c = (double)__popc(f);
        re = fma(c, d.wr[g], re);
        im = fma(c, d.wi[g], im);
    }
    return re;
}

// One thread per output index.  Bound by the vector-memory address path: a partner costs one
// 16-byte gather (16 cycles a wave) beside its arithmetic, so the two half tables sit in LDS
// (rank as 16 bits) and not in three dependent global reads a partner, and SEC_U partners are in
// flight at a time.  v0 = y v0 + H (x v1) with the optional device factors xs, ys.  REAL: no
// coefficient and no diagonal weight has an imaginary part (their products are left out).
// N=24 at k=12 (2704156 states, Heisenberg), us a call: 154 -> 108; N=28 at k=14 2632 -> 1740.
constexpr int SEC_U = 4;
template <bool REAL, bool LDS, int TPB>
__global__ __launch_bounds__(TPB) void hv_sector_kernel(const double2 *__restrict__ v1, double2 *__restrict__ v0,
                                                        const uint32_t *__restrict__ list1,
                                                        const uint32_t *__restrict__ rank,
                                                        const uint32_t *__restrict__ offset,
                                                        const SectorTerm *__restrict__ terms, int nterm,
                                                        const DiagDev *__restrict__ diagp, int ihf, int ihf0,
                                                        double shift, int fresh, uint64_t dim,
                                                        const double *__restrict__ xs, const double *__restrict__ ys,
                                                        double *__restrict__ partial)
{
    extern __shared__ uint32_t sec_smem[];
    __shared__ double red[2 * TPB];
    const int tid = threadIdx.x;
    const uint32_t right = (1u << ihf) - 1u;
    uint32_t *off = sec_smem;
    uint16_t *rk = reinterpret_cast<uint16_t *>(sec_smem + (LDS ? (1u << ihf0) : 0u));
    if (LDS) {
        for (uint32_t i = tid; i < (1u << ihf0); i += TPB) off[i] = offset[i];
        for (uint32_t i = tid; i <= right; i += TPB) rk[i] = (uint16_t)rank[i];
        __syncthreads();
    }
    const DiagDev &dg = *diagp;
    const double x_s = xs ? *xs : 1.0, y_s = ys ? *ys : 1.0;
    double pr_re = 0.0, pr_im = 0.0;
    const uint64_t stride = (uint64_t)TPB * gridDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * TPB + tid; i < dim; i += stride) {
        const uint32_t s = list1[i];
        const double2 x = v1[i];
        double di = 0.0, dr;
        if (REAL) {
            dr = dg.c0r;
            for (int g = 0; g < dg.ngroups; ++g) {
                const uint32_t f = (dg.kind[g] == 0) ? (s & dg.mask[g]) : ((s ^ (s >> dg.shift[g])) & dg.mask[g]);
                dr = fma((double)__popc(f), dg.wr[g], dr);
            }
        } else {
            dr = sector_diag(dg, s, di);
        }
        dr += shift;
        double ar = dr * x.x, ai = dr * x.y;
        if (!REAL) {
            ar = dr * x.x - di * x.y;
            ai = dr * x.y + di * x.x;
        }
        for (int t = 0; t < nterm; t += SEC_U) {
            double2 y[SEC_U];
#pragma unroll
            for (int u = 0; u < SEC_U; ++u) {
                const uint32_t m = terms[t + u].mask;   // (padded with zero masks: never active)
                const uint32_t p = s ^ m;
                y[u] = make_double2(0.0, 0.0);
                if (__popc(s & m) == 1) {   // else the partner lies outside the sector: coefficient 0
                    const uint32_t at = LDS ? off[p >> ihf] + rk[p & right] : offset[p >> ihf] + rank[p & right];
                    y[u] = v1[at];
                }
            }
#pragma unroll
            for (int u = 0; u < SEC_U; ++u) {
                // an active partner's selector is odd (see sector_terms): c1
                const double cr = terms[t + u].c1r, ci = terms[t + u].c1i;
                if (REAL) {
                    ar = fma(cr, y[u].x, ar);
                    ai = fma(cr, y[u].y, ai);
                } else {
                    ar = fma(cr, y[u].x, fma(-ci, y[u].y, ar));
                    ai = fma(cr, y[u].y, fma(ci, y[u].x, ai));
                }
            }
        }
        ar *= x_s;
        ai *= x_s;
        pr_re += x.x * ar + x.y * ai;
        pr_im += x.x * ai - x.y * ar;
        double2 o = make_double2(ar, ai);
        if (!fresh) {
            const double2 old = v0[i];
            o = make_double2(fma(y_s, old.x, ar), fma(y_s, old.y, ai));
        }
        v0[i] = o;
    }
    red[2 * tid] = pr_re;
    red[2 * tid + 1] = pr_im;
    __syncthreads();
    for (int st = TPB / 2; st > 0; st >>= 1) {
        if (tid < st) {
            red[2 * tid] += red[2 * (tid + st)];
            red[2 * tid + 1] += red[2 * (tid + st) + 1];
        }
        __syncthreads();
    }
    if (tid == 0) {
        partial[2 * blockIdx.x] = red[0];
        partial[2 * blockIdx.x + 1] = red[1];
    }
}

// intalv_xy (S_one_half/Hybrid_TPS_DSF.f90:89-193) as a gather: one thread per target
// index l (sector k + ipm) sums e^{i q.r_j} x(source index of t with bit j flipped) over
// the bits j of its state t that ipm has just set (ipm = +1) or cleared (-1), in ascending
// j -- per element, the order in which the reference's site-outer scatter adds them.
struct XyArgs {
    int n, ipm;
    double phr[32], phi[32];
};

__global__ __launch_bounds__(256) void k_intalv_xy(const double2 *__restrict__ x, double2 *__restrict__ v,
                                                   const uint32_t *__restrict__ list1_dst,
                                                   const uint32_t *__restrict__ rank,
                                                   const uint32_t *__restrict__ offset_src, XyArgs a, int ihf,
                                                   uint64_t dim)
{
    const uint32_t right = (1u << ihf) - 1u;
    const uint64_t stride = (uint64_t)blockDim.x * gridDim.x;
    for (uint64_t l = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; l < dim; l += stride) {
        const uint32_t t = list1_dst[l];
        double ar = 0.0, ai = 0.0;
        for (int j = 0; j < a.n; ++j) {
            if ((int)((t >> j) & 1u) != (a.ipm > 0 ? 1 : 0)) continue;
            const uint32_t s = t ^ (1u << j);
            const double2 y = x[(uint64_t)rank[s & right] + (uint64_t)offset_src[s >> ihf]];
            ar += a.phr[j] * y.x - a.phi[j] * y.y;
            ai += a.phi[j] * y.x + a.phr[j] * y.y;
        }
        v[l] = make_double2(ar, ai);
    }
}

int intalv_xy_apply(pned_ctx *ctx, const pned_vec *x, pned_vec *v, const double *qv, const double *site_vec,
                    int ipm)
{
    const pned_ctx *src = x->ctx;
    if (v->ctx != ctx) return fail(PNED_E_ARG, "v must belong to the target context");
    if (ctx->q != 2 || !src || src->q != 2 || src->n != ctx->n)
        return fail(PNED_E_ARG, "S^+(q): two S=1/2 contexts of the same cluster");
    if (ctx->sector_k < 0 || src->sector_k < 0 || ctx->sector_k != src->sector_k + ipm)
        return fail(PNED_E_ARG, "S^+/-(q): x in the sector with k set bits, v in the one with k + ipm");
    if (src->device != ctx->device) return fail(PNED_E_ARG, "S^+(q): both contexts on one device");
    if (x->nvec != 1 || v->nvec != 1 || x->dtype != PNED_C128 || v->dtype != PNED_C128)
        return fail(PNED_E_UNSUPPORTED, "S^+(q) takes one complex128 column");
    XyArgs a{};
    a.n = ctx->n;
    a.ipm = ipm;
    for (int j = 0; j < ctx->n; ++j) {
        const double qn = qv[0] * site_vec[2 * j] + qv[1] * site_vec[2 * j + 1];
        a.phr[j] = std::cos(qn);
        a.phi[j] = std::sin(qn);
    }
    // x was written on the source context's stream
    PNED_HIP(hipStreamSynchronize(src->stream));
    const uint64_t dim = (uint64_t)ctx->dim;
    const int grid = (int)std::min<uint64_t>((dim + 255) / 256, 8192);
    hipLaunchKernelGGL(k_intalv_xy, dim3(grid), dim3(256), 0, ctx->stream, (const double2 *)x->data,
                       (double2 *)v->data, ctx->d_list1, src->d_srank, src->d_soffset, a, (ctx->n + 1) / 2, dim);
    PNED_HIP(hipGetLastError());
    return PNED_OK;
}


void free_sector(pned_ctx *ctx)
{
    if (ctx->d_list1) (void)hipFree(ctx->d_list1);
    if (ctx->d_srank) (void)hipFree(ctx->d_srank);
    if (ctx->d_soffset) (void)hipFree(ctx->d_soffset);
    if (ctx->d_sterms) (void)hipFree(ctx->d_sterms);
    ctx->d_list1 = ctx->d_srank = ctx->d_soffset = nullptr;
    ctx->d_sterms = nullptr;
    ctx->sector_k = -1;
    ctx->sector_nterm = 0;
}

// the two-bit flip terms of the decomposition, or an error if the operator moves states
// out of the sector (a one-bit flip, or a two-bit flip of aligned spins)
static int sector_terms(const S12Plan &pl, std::vector<SectorTerm> &out)
{
    out.clear();
    for (const Term &t : pl.terms) {
        const bool zero0 = t.c0r == 0.0 && t.c0i == 0.0, zero1 = t.c1r == 0.0 && t.c1i == 0.0;
        if (zero0 && zero1) continue;
        const int nb = __builtin_popcount(t.gmask);
        // aligned spins (the only states a two-bit flip takes out of the sector) select
        // c0 when the selector is exactly the two flipped bits
        if (nb != 2 || t.selmask != t.gmask || !zero0)
            return fail(PNED_E_UNSUPPORTED, "the operator does not conserve S^z (no sector basis)");
        out.push_back(SectorTerm{t.gmask, t.selmask, t.c0r, t.c0i, t.c1r, t.c1i});
    }
    return PNED_OK;
}

// device copy of the terms, padded to whole batches with terms that never apply
static int upload_sector_terms(pned_ctx *ctx, std::vector<SectorTerm> st)
{
    ctx->sector_nterm = (int)st.size();
    ctx->sector_real = (ctx->s12.c0i == 0.0) ? 1 : 0;
    for (const SectorTerm &t : st)
        if (t.c1i != 0.0) ctx->sector_real = 0;
    for (const DiagGroup &g : ctx->s12.diag)
        if (g.wi != 0.0) ctx->sector_real = 0;
    st.resize((st.size() / SEC_U + 1) * SEC_U, SectorTerm{0, 0, 0.0, 0.0, 0.0, 0.0});
    PNED_HIP(hipStreamSynchronize(ctx->stream));
    if (ctx->d_sterms) PNED_HIP(hipFree(ctx->d_sterms));
    ctx->d_sterms = nullptr;
    PNED_HIP(hipMalloc(&ctx->d_sterms, sizeof(SectorTerm) * st.size()));
    PNED_HIP(hipMemcpy(ctx->d_sterms, st.data(), sizeof(SectorTerm) * st.size(), hipMemcpyHostToDevice));
    return PNED_OK;
}

int refresh_sector_terms(pned_ctx *ctx)
{
    std::vector<SectorTerm> st;
    PNED_TRY(sector_terms(ctx->s12, st));
    return upload_sector_terms(ctx, st);
}

int launch_hv_sector(pned_ctx *ctx, const pned_vec *v1, pned_vec *v0, double eperbd, bool fresh, double *prdct_host,
                     const double *d_xs, const double *d_ys)
{
    if (v1->nvec != 1 || v1->dtype != PNED_C128)
        return fail(PNED_E_UNSUPPORTED, "sector H.v takes one complex128 column");
    // the diagonal table is shared with the full-space path
    PNED_TRY(ensure_s12_plan(ctx, 0, PNED_C128));
    const uint64_t dim = (uint64_t)ctx->dim;
    const int ihf = (ctx->n + 1) / 2, ihf0 = ctx->n / 2;
    // tables in LDS up to 28 sites (98 KB), from L2 above.  1024 threads share one copy from 21 sites on,
    // on a grid of resident blocks that stage it once (512; 256 at 27 and 28 sites, where one block fills a
    // CU's LDS).  us a call at k of 24 sites, 1024 threads and 256: k=12 103 and 135, k=7 35 and 49, k=3 27
    // and 29; 26 sites, k=6 28 and 42, k=3 26 and 31; 28 sites, k=6 in a second, partial round of blocks 51,
    // resident 48 (k=14 1635 and 1649); 20 sites, k=10 27 and 27, 16 sites, k=8 25.1 and 24.6.
    const size_t tab = (sizeof(uint32_t) << ihf0) + (sizeof(uint16_t) << ihf);
    const bool lds = ihf <= 14;
    const int tpb = lds && ihf >= 11 ? 1024 : 256;
    const uint64_t cap = tpb == 256 ? 4096 : ihf == 14 ? 256 : 512;
    const int grid = (int)std::min<uint64_t>((dim + tpb - 1) / tpb, cap);
    PNED_TRY(ensure_partial(ctx, 2 * (size_t)grid));
    PNED_TRY(ensure_result(ctx, 8));
    auto launch = [&](auto k) -> int {
        PNED_HIP(hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize,
                                     (int)(lds ? tab : 0)));
        hipLaunchKernelGGL(k, dim3(grid), dim3(tpb), lds ? tab : 0, ctx->stream, (const double2 *)v1->data,
                           (double2 *)v0->data, ctx->d_list1, ctx->d_srank, ctx->d_soffset,
                           (const SectorTerm *)ctx->d_sterms, ctx->sector_nterm, ctx->d_diag, ihf, ihf0,
                           -(double)ctx->ibond * eperbd, fresh ? 1 : 0, dim, d_xs, d_ys, ctx->d_partial);
        PNED_HIP(hipGetLastError());
        return PNED_OK;
    };
    const bool real = ctx->sector_real != 0;
    if (tpb == 1024) PNED_TRY(real ? launch(hv_sector_kernel<true, true, 1024>) : launch(hv_sector_kernel<false, true, 1024>));
    else if (lds) PNED_TRY(real ? launch(hv_sector_kernel<true, true, 256>) : launch(hv_sector_kernel<false, true, 256>));
    else PNED_TRY(real ? launch(hv_sector_kernel<true, false, 256>) : launch(hv_sector_kernel<false, false, 256>));
    PNED_TRY(reduce_rows_result(ctx, grid, 2));
    if (prdct_host) {
        PNED_HIP(hipMemcpyAsync(ctx->h_result, ctx->d_result, 2 * sizeof(double), hipMemcpyDeviceToHost,
                                ctx->stream));
        PNED_HIP(hipStreamSynchronize(ctx->stream));
        prdct_host[0] = ctx->h_result[0];
        prdct_host[1] = ctx->h_result[1];
    }
    return PNED_OK;
}

}  // namespace pned

using namespace pned;

extern "C" int pned_ctx_sz_sector(pned_ctx *ctx, int n_down)
{
    if (!ctx) return fail(PNED_E_ARG, "null context");
    if (ctx->q != 2) return fail(PNED_E_UNSUPPORTED, "sector basis: S=1/2 only");
    PNED_HIP(hipSetDevice(ctx->device));
    PNED_HIP(hipStreamSynchronize(ctx->stream));
    const int n = ctx->n;
    if (n_down < 0) {   // back to the full 2^N space
        free_sector(ctx);
        ctx->dim = (int64_t)1 << n;
        return PNED_OK;
    }
    if (n_down > n) return fail(PNED_E_ARG, "#(E02A)# Incorrect ldim or n given to sz");
    if (n > 32) return fail(PNED_E_UNSUPPORTED, "sector basis: N <= 32");
    PNED_TRY(reset_layout(ctx));   // the sector tables index basis states directly
    std::vector<SectorTerm> st;
    PNED_TRY(sector_terms(ctx->s12, st));
    const int ihf = (n + 1) / 2, ihf0 = n / 2;
    // binomials and the two half tables
    std::vector<std::vector<uint64_t>> C(33, std::vector<uint64_t>(33, 0));
    for (int a = 0; a <= 32; ++a) {
        C[a][0] = 1;
        for (int b = 1; b <= a; ++b) C[a][b] = C[a - 1][b - 1] + (b <= a - 1 ? C[a - 1][b] : 0);
    }
    std::vector<uint32_t> rank((size_t)1 << ihf), offset((size_t)1 << ihf0);
    {
        std::vector<uint32_t> seen(ihf + 1, 0);
        for (uint64_t r = 0; r < ((uint64_t)1 << ihf); ++r) rank[r] = seen[__builtin_popcountll(r)]++;
    }
    uint64_t total = 0;
    for (uint64_t l = 0; l < ((uint64_t)1 << ihf0); ++l) {
        offset[l] = (uint32_t)total;
        const int need = n_down - __builtin_popcountll(l);
        if (need >= 0 && need <= ihf) total += C[ihf][need];
    }
    if (total < 3) return fail(PNED_E_ARG, "#(E02A)# Incorrect ldim or n given to sz");
    if (total > 0xFFFFFFFFull) return fail(PNED_E_UNSUPPORTED, "sector larger than 2^32 states");
    std::vector<uint32_t> list1(total);
    {
        uint64_t i = 0;
        for (uint64_t l = 0; l < ((uint64_t)1 << ihf0); ++l)
            for (uint64_t r = 0; r < ((uint64_t)1 << ihf); ++r)
                if (__builtin_popcountll(l) + __builtin_popcountll(r) == n_down)
                    list1[i++] = (uint32_t)((l << ihf) | r);
    }
    free_sector(ctx);
    PNED_HIP(hipMalloc((void **)&ctx->d_list1, sizeof(uint32_t) * list1.size()));
    PNED_HIP(hipMalloc((void **)&ctx->d_srank, sizeof(uint32_t) * rank.size()));
    PNED_HIP(hipMalloc((void **)&ctx->d_soffset, sizeof(uint32_t) * offset.size()));
    PNED_HIP(hipMemcpy(ctx->d_list1, list1.data(), sizeof(uint32_t) * list1.size(), hipMemcpyHostToDevice));
    PNED_HIP(hipMemcpy(ctx->d_srank, rank.data(), sizeof(uint32_t) * rank.size(), hipMemcpyHostToDevice));
    PNED_HIP(hipMemcpy(ctx->d_soffset, offset.data(), sizeof(uint32_t) * offset.size(), hipMemcpyHostToDevice));
    PNED_TRY(upload_sector_terms(ctx, st));
    ctx->sector_k = n_down;
    ctx->dim = (int64_t)total;
    return PNED_OK;
}
