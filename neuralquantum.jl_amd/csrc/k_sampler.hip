// Metropolis-Hastings with LocalRule on the doubled (row, column) space,
// p(s, e) ∝ |rho(s, e)|^2, log p = 2 Re log rho (base_batched_networks.jl:255-258).
//
// Schedule (Metropolis.jl:101-167, BaseIterativeSampler.jl:5-17): optional
// restart from a uniform configuration, `burn` calls of `passes` proposals,
// then one stored slice after each further call of `passes` proposals.  A
// proposal flips one uniformly chosen doubled site (LocalRule.jl:30-38) and is
// rejected iff u - exp(log p' - log p) >= 0 (Metropolis.jl:148-154).
//
// Mapping: a group of `lpc` lanes (power of two) runs one chain, 64/lpc chains
// per wavefront.  Lane g of a group owns lambda units h = g + lpc r (both
// sides) and Pi units a = g + lpc r; only the lambda and Pi blocks enter
// Re log rho, the mu block does not.  The effective angles stay in registers;
// a proposal costs one FMA + one f (softplus or logcosh, the NDM's activation)
// per lambda unit of the flipped side and one complex update + Re f per Pi
// unit, then a group reduction.
// Angles are recomputed from the configuration at the start of every call so
// incremental rounding never accumulates over more than `passes` updates.
// Random numbers: Philox4x32-10, counter (t, iteration, chain, 1) for proposal
// t; each lane of the group draws for one future proposal and the draws are
// shuffled to the group when used.
#include <algorithm>

#include "nq_device.h"
#include "nq_kernels.h"

namespace {

template <typename T>
__device__ __forceinline__ T xv(uint32_t bits, int i) { return ((bits >> i) & 1u) ? T(1) : T(-1); }

// the block body; bx = the workgroup's number in its problem's grid
template <typename T, int US, int ACT>
__device__ __forceinline__ void metropolis_body(const samp_args& a, int bx) {
    extern __shared__ __align__(16) unsigned char smem[];
    const ndm_dims d = a.d;
    const int N = d.N, nh = d.nh, na = d.na;
    T* sp = reinterpret_cast<T*>(smem);
    const T* gp = reinterpret_cast<const T*>(a.p);
    for (int k = threadIdx.x; k < d.np; k += blockDim.x) sp[k] = gp[k];
    __syncthreads();

    const int lpc = a.lpc;
    const int lane = threadIdx.x & 63;
    const int g = lane & (lpc - 1);
    // the chain's lanes: rep copies of the group (FP64), which share the random draws
    const int width = lpc * a.rep;
    const int gw = lane & (width - 1);
    const int gbase = lane - g;
    const int cpw = 64 / width;
    const int64_t wave_glob = (int64_t)bx * (blockDim.x >> 6) + (threadIdx.x >> 6);
    const int64_t chain = wave_glob * cpw + lane / width;
    const bool live = chain < a.chains;
    const uint32_t pmask = (N >= 32) ? 0xffffffffu : ((1u << N) - 1u);
    const uint32_t k0 = (uint32_t)a.seed, k1 = (uint32_t)(a.seed >> 32);
    const uint32_t iter = a.iter_dev ? *a.iter_dev : a.iter;
    const T half = T(0.5);

    const bool diag = a.diag != 0;
    const uint32_t ctr3 = 16u * a.tag;
    uint64_t key = 0;
    if (live) {
        if (a.restart) {
            philox_out o = philox4x32_10(0u, iter, (uint32_t)chain, ctr3, k0, k1);
            if (diag) {
                const uint64_t s = ((uint64_t)o.x[0] | ((uint64_t)o.x[1] << 32)) & (uint64_t)pmask;
                key = s | (s << N);
            } else {
                const uint64_t m2 = (2 * N >= 64) ? ~0ull : ((1ull << (2 * N)) - 1ull);
                key = ((uint64_t)o.x[0] | ((uint64_t)o.x[1] << 32)) & m2;
            }
        } else {
            key = a.chain_state[chain];
        }
    }

    T th_s[US], th_e[US], f_s[US], f_e[US], fpi[US];
    cplx<T> z[US];
    uint64_t acc = 0;
    uint32_t t = a.t0;
    uint32_t rx0 = 0, rx1 = 0, rx2 = 0;   // this lane's pre-drawn proposal
    const int calls = a.burn + a.stored;

    for (int call = 0; call < calls; ++call) {
        // refresh the angles from the configuration
        const uint32_t ks = (uint32_t)key & pmask, ke = (uint32_t)(key >> N) & pmask;
#pragma unroll
        for (int r = 0; r < US; ++r) {
            const int h = g + lpc * r;
            th_s[r] = th_e[r] = f_s[r] = f_e[r] = fpi[r] = T(0);
            z[r] = cmk(T(0), T(0));
            if (h < nh) {
                T ts = sp[d.hla + h], te = ts;
                for (int i = 0; i < N; ++i) {
                    const T w = sp[d.wla + h + nh * i];
                    ts += w * xv<T>(ks, i);
                    te += w * xv<T>(ke, i);
                }
                th_s[r] = ts; th_e[r] = te;
                f_s[r] = act_f<ACT>(ts); f_e[r] = act_f<ACT>(te);
            }
            if (h < na) {
                T zr = sp[d.dla + h], zi = T(0);
                for (int i = 0; i < N; ++i) {
                    const T xs = xv<T>(ks, i), xe = xv<T>(ke, i);
                    zr += half * sp[d.ula + h + na * i] * (xs + xe);
                    zi += half * sp[d.umu + h + na * i] * (xs - xe);
                }
                z[r] = cmk(zr, zi);
                fpi[r] = cact_re<ACT>(z[r]);
            }
        }
        for (int q = 0; q < a.passes; ++q, ++t) {
            const int slot = (int)((t - a.t0) % (uint32_t)lpc);
            if (slot == 0) {
                philox_out o = philox4x32_10(t + (uint32_t)g, iter, (uint32_t)chain, ctr3 + 1u, k0, k1);
                rx0 = o.x[0]; rx1 = o.x[1]; rx2 = o.x[2];
            }
            const uint32_t x0 = __shfl(rx0, gbase + slot, 64);
            const uint32_t x1 = __shfl(rx1, gbase + slot, 64);
            const uint32_t x2 = __shfl(rx2, gbase + slot, 64);
            // diagonal chain: site j flipped in sigma and eta, log p = Re log rho(sigma, sigma)
            const int site = (int)(((uint64_t)x0 * (uint64_t)(diag ? N : 2 * N)) >> 32);
            const bool col = site >= N;
            const int j = col ? site - N : site;
            const uint32_t bits = col ? (uint32_t)(key >> N) : (uint32_t)key;
            const T c = ((bits >> j) & 1u) ? T(-2) : T(2);

            T delta = T(0);
            T nth[US], nf[US], nfpi[US];
            cplx<T> nz[US];
#pragma unroll
            for (int r = 0; r < US; ++r) {
                const int h = g + lpc * r;
                nth[r] = nf[r] = nfpi[r] = T(0);
                nz[r] = z[r];
                if (h < nh) {
                    const T th = col ? th_e[r] : th_s[r];
                    nth[r] = th + c * sp[d.wla + h + nh * j];
                    nf[r] = act_f<ACT>(nth[r]);
                    delta += nf[r] - (col ? f_e[r] : f_s[r]);
                }
                if (h < na) {
                    const T cu = diag ? c : c * half;
                    nz[r].re += cu * sp[d.ula + h + na * j];
                    if (!diag) nz[r].im += (col ? -cu : cu) * sp[d.umu + h + na * j];
                    nfpi[r] = cact_re<ACT>(nz[r]);
                    delta += (diag ? T(1) : T(2)) * (nfpi[r] - fpi[r]);
                }
            }
            delta = group_total(delta, lpc);
            delta += c * sp[d.bla + j];

            bool accept;
            if constexpr (sizeof(T) == 8) {
                const double u = u01_53(x1, x2);
                accept = !(u - exp((double)delta) >= 0.0);
            } else {
                const float u = u01_24(x1);
                accept = !(u - expf((float)delta) >= 0.0f);
            }
            if (accept && live) {
                key ^= diag ? ((1ull << site) | (1ull << (site + N))) : (1ull << site);
                ++acc;
#pragma unroll
                for (int r = 0; r < US; ++r) {
                    const int h = g + lpc * r;
                    if (h < nh) {
                        if (diag) { th_s[r] = th_e[r] = nth[r]; f_s[r] = f_e[r] = nf[r]; }
                        else if (col) { th_e[r] = nth[r]; f_e[r] = nf[r]; }
                        else { th_s[r] = nth[r]; f_s[r] = nf[r]; }
                    }
                    if (h < na) { z[r] = nz[r]; fpi[r] = nfpi[r]; }
                }
            }
        }
        if (call >= a.burn && live && gw == 0 && a.samples) {
            const int slice = a.slice0 + call - a.burn;
            a.samples[chain + (int64_t)slice * a.chains] = key;
        }
    }
    if (live && gw == 0) {
        if (a.chain_state) a.chain_state[chain] = key;
        if (a.compat_stale_last_slice && a.samples)
            a.samples[chain + (int64_t)(a.stored) * a.chains] = 0ull;   // defect D1: slice L stays at the fill
        if (a.accepted) atomicAdd(a.accepted, (unsigned long long)acc);
        if (a.chain_acc) a.chain_acc[chain] += (uint32_t)acc;   // one lane per chain: no race
    }
}

// ---- FP64: the same chains without a transcendental function per proposal
// Over the units the acceptance ratio e^(dlog p) is a ratio of products:
//   softplus  e^f(x) = 1 + e^x,  e^(2 Re f(z)) = |1 + e^z|^2
//   logcosh   e^f(x) = e^-x (1 + e^2x) / 2,  e^(2 Re f(z)) = e^(-2 Re z) |1 + e^2z|^2 / 4
// with e^(K x) (K = 1 or 2) multiplied by a table entry e^(+-2 K w) when a site flips, and the
// factors e^-x, which are linear in the flip, taken into the visible bias of the flipped site.
// A lane keeps k e^(K theta) of its lambda units (both sides) and k e^(K z) of its Pi units; the
// group keeps the products over its units of k (1 + e^(K theta)) per side (Gs, Ge) and of
// k^2 |1 + e^(K z)|^2 (Gp).  A proposal multiplies, adds 1, reduces two products over the group
// and accepts by u Gs Gp < Gs' Gp' e^(bias): a handful of FMAs per unit where exp, log1p and
// sincos took about 700 instructions.  What is left is a chain of dependent FP64 operations and two
// group reductions per proposal.  Per launch, before and now: 4x4 XYZ, 4096 chains, 1782 proposals
// 4.17 -> 0.84 ms; 12 sites, 1024 chains, 1650 proposals 2.53 -> 0.52 ms; 6 sites, 16 chains, 2925
// proposals 4.49 -> 0.81 ms.
//
// The constants k = e^(-m / 2), m the largest |K theta| a unit can reach, centre every factor; the
// sum of the ranges over the units bounds every product over them.  That does not bound a unit alone:
// its kept factor goes from e^(-1.5 m) to e^(m / 2) and its table entries reach e^(+-2 m), so every
// unit also stays within m <= kUnitRange.  Where a unit leaves that, the sum leaves e^(+-kRatioRange),
// or a bias e^(+-kRatioBias), the chains run through metropolis_body instead, in about the former times
// (4x4 XYZ 4.2 ms).  With N = 16, nh = na = 32 the sum does so at a mean |w| of about 0.65 (softplus) or
// 0.33 (logcosh).
// Rounding of the kept factors: one product per accepted flip, set again from the configuration
// at least every kRatioRefresh proposals or every call, whichever is longer.
constexpr double kRatioRange = 600.0, kUnitRange = 300.0, kRatioBias = 60.0;
constexpr int kRatioRefresh = 64;

// LDS bytes of the tables: e^(+-2 K w) per (site, lambda unit), two complex factors per (site, Pi
// unit), e^(+-2 b) per site
__host__ __device__ inline size_t ratio_lds_bytes(const ndm_dims& d) {
    return 16 * (size_t)d.N * ((size_t)d.nh + 2 * (size_t)d.na + 1);
}

// runs the workgroup's chains and returns true, or returns false (before anything is written)
// where the weights leave the range
template <int LPC, int US, int ACT, bool DIAG>
__device__ __forceinline__ bool metropolis_ratio_body(const samp_args& a, int bx) {
    extern __shared__ __align__(16) unsigned char smem[];
    const ndm_dims d = a.d;
    const int N = d.N, nh = d.nh, na = d.na;
    const double* gp = reinterpret_cast<const double*>(a.p);
    constexpr bool diag = DIAG;
    constexpr double K = ACT == NQ_ACT_LOGCOSH ? 2.0 : 1.0;
    double2* tl = reinterpret_cast<double2*>(smem);            // [j nh + h] e^(2 K w), e^(-2 K w)
    double2* tp = tl + N * nh;                                 // [j na + a] factor of a flip to +1
    double2* tm = tp + N * na;                                 //            of a flip to -1
    double2* tb = tm + N * na;                                 // [j] e^(2 b), e^(-2 b)

    constexpr int lpc = LPC;
    const int lane = threadIdx.x & 63;
    const int g = lane & (lpc - 1);
    // the chain's lanes: rep copies of the group run it side by side and share its random draws
    const int width = lpc * a.rep;
    const int gw = lane & (width - 1);
    const int gbase = lane - gw;

    // this lane's units: the centring constants, the factors with every site at -1 (e0, and w0,
    // which is real there), and the range of the group's products
    int hu[US], au[US];
    double kl[US], kp[US], e0[US], w0[US], range = 0.0;
#pragma unroll
    for (int r = 0; r < US; ++r) {
        const int u = g + lpc * r;
        hu[r] = u < nh ? u : -1;
        au[r] = u < na ? u : -1;
        kl[r] = kp[r] = 1.0;
        e0[r] = w0[r] = 0.0;
        if (hu[r] >= 0) {
            double t = gp[d.hla + u], m = fabs(t);
            for (int i = 0; i < N; ++i) {
                const double w = gp[d.wla + u + nh * i];
                t -= w;
                m += fabs(w);
            }
            kl[r] = exp(-0.5 * K * m);
            e0[r] = exp(K * t - 0.5 * K * m);
            range += K * m <= kUnitRange ? 0.5 * K * m + 0.7 : HUGE_VAL;
        }
        if (au[r] >= 0) {
            double t = gp[d.dla + u], m = fabs(t);
            for (int i = 0; i < N; ++i) {
                const double w = gp[d.ula + u + na * i];
                t -= w;
                m += fabs(w);
            }
            kp[r] = exp(-0.5 * K * m);
            w0[r] = exp(K * t - 0.5 * K * m);
            range += K * m <= kUnitRange ? K * m + 1.4 : HUGE_VAL;
        }
    }
    range = group_total(range, lpc);
    // the flipped site's bias factor: the visible bias, for logcosh less the units' linear parts
    bool ok = range <= kRatioRange;
    for (int j = 0; j < N; ++j) {
        double b = gp[d.bla + j];
        if constexpr (ACT == NQ_ACT_LOGCOSH) {
            double lin = 0.0;
#pragma unroll
            for (int r = 0; r < US; ++r) {
                if (hu[r] >= 0) lin += gp[d.wla + hu[r] + nh * j];
                if (au[r] >= 0) lin += gp[d.ula + au[r] + na * j];
            }
            b -= group_total(lin, lpc);
        }
        ok = ok && 2.0 * fabs(b) <= kRatioBias;
        if (threadIdx.x == 0) tb[j] = make_double2(exp(2.0 * b), exp(-2.0 * b));
    }
    if (!__builtin_amdgcn_readfirstlane((int)ok)) return false;   // the same sums in every group
    for (int k = threadIdx.x; k < N * nh; k += blockDim.x) {
        const double w = 2.0 * K * gp[d.wla + k];
        tl[k] = make_double2(exp(w), exp(-w));
    }
    for (int k = threadIdx.x; k < N * na; k += blockDim.x) {
        // a flip of one side to v moves z by v (u_la +- i u_mu); on the diagonal both sides flip
        const double ul = (diag ? 2.0 : 1.0) * K * gp[d.ula + k];
        const double um = diag ? 0.0 : K * gp[d.umu + k];
        double s, c;
        sincos(um, &s, &c);
        const double ep = exp(ul), em = exp(-ul);
        tp[k] = make_double2(ep * c, ep * s);
        tm[k] = make_double2(em * c, -em * s);
    }
    __syncthreads();

    const int cpw = 64 / width;
    const int64_t wave_glob = (int64_t)bx * (blockDim.x >> 6) + (threadIdx.x >> 6);
    const int64_t chain = wave_glob * cpw + lane / width;
    const bool live = chain < a.chains;
    const uint32_t pmask = (N >= 32) ? 0xffffffffu : ((1u << N) - 1u);
    const uint32_t k0 = (uint32_t)a.seed, k1 = (uint32_t)(a.seed >> 32);
    const uint32_t iter = a.iter_dev ? *a.iter_dev : a.iter;
    const uint32_t ctr3 = 16u * a.tag;
    uint64_t key = 0;
    if (live) {
        if (a.restart) {
            const philox_out o = philox4x32_10(0u, iter, (uint32_t)chain, ctr3, k0, k1);
            if (diag) {
                const uint64_t s = ((uint64_t)o.x[0] | ((uint64_t)o.x[1] << 32)) & (uint64_t)pmask;
                key = s | (s << N);
            } else {
                const uint64_t m2 = (2 * N >= 64) ? ~0ull : ((1ull << (2 * N)) - 1ull);
                key = ((uint64_t)o.x[0] | ((uint64_t)o.x[1] << 32)) & m2;
            }
        } else {
            key = a.chain_state[chain];
        }
    }

    double es[US], ee[US], wr[US], wi[US];   // k e^(K theta) of the row and column side, k e^(K z)
    double Gs = 1.0, Ge = 1.0, Gp = 1.0;
    uint32_t acc = 0;
    const uint32_t nsite = (uint32_t)(diag ? N : 2 * N);
    // Each lane draws one future proposal (site, uniform) of its chain and hands it over when its
    // turn comes.  Three stages keep the LDS round trips off the chain of dependent products: the
    // hand-over two proposals ahead, the table entries of its site one ahead.
    int dsite = 0;
    double du = 0.0;
    auto hand_over = [&](uint32_t q, int& site, double& u) {
        const int slot = (int)(q & (uint32_t)(width - 1));
        if (slot == 0) {
            const philox_out o = philox4x32_10(a.t0 + q + (uint32_t)gw, iter, (uint32_t)chain, ctr3 + 1u, k0, k1);
            dsite = (int)(((uint64_t)o.x[0] * (uint64_t)nsite) >> 32);
            du = u01_53(o.x[1], o.x[2]);
        }
        site = __shfl(dsite, gbase + slot, 64);
        u = __shfl(du, gbase + slot, 64);
    };
    // table entries of one flip; the direction is that of the configuration before the proposal
    // in between, so they are loaded again on the rare step whose site that proposal flipped
    struct flip { int site; double u; bool down; double l[US], fr[US], fi[US], b; };
    auto load = [&](flip& f) {
        const bool col = !diag && f.site >= N;
        const int j = col ? f.site - N : f.site;
        f.down = ((key >> f.site) & 1ull) != 0;        // the flip takes +1 to -1
        const double2* t2 = f.down ? tm : tp;
        const int o = f.down ? 1 : 0;
#pragma unroll
        for (int r = 0; r < US; ++r) {
            f.l[r] = reinterpret_cast<const double*>(tl)[2 * (j * nh + (hu[r] < 0 ? 0 : hu[r])) + o];
            const double2 w = t2[j * na + (au[r] < 0 ? 0 : au[r])];
            f.fr[r] = w.x;
            f.fi[r] = col ? -w.y : w.y;
        }
        f.b = reinterpret_cast<const double*>(tb)[2 * j + o];
    };
    flip f0, f1;
    hand_over(0u, f0.site, f0.u);
    load(f0);
    hand_over(1u, f1.site, f1.u);

    uint32_t q = 0;
    // proposal q: f; f's place then takes proposal q + 2's site and uniform
    auto step = [&](flip& f, flip& next) {
        if (__any(f.down != (((key >> f.site) & 1ull) != 0))) load(f);
        load(next);
        int site2;
        double u2;
        hand_over(q + 2u, site2, u2);
        ++q;
        const bool col = !diag && f.site >= N;
        double ne[US], nr[US], ni[US], ll = 1.0, lp = 1.0;
#pragma unroll
        for (int r = 0; r < US; ++r) {
            ne[r] = (col ? ee[r] : es[r]) * f.l[r];
            ll *= kl[r] + ne[r];
            nr[r] = wr[r] * f.fr[r] - wi[r] * f.fi[r];
            ni[r] = wr[r] * f.fi[r] + wi[r] * f.fr[r];
            const double dr = kp[r] + nr[r];
            lp *= diag ? dr : dr * dr + ni[r] * ni[r];
        }
        const double nl = group_product<LPC>(ll), np = group_product<LPC>(lp);
        const bool accept = !(f.u * ((col ? Ge : Gs) * Gp) - nl * np * f.b >= 0.0);
        const bool as = accept && !col, ae = accept && (col || diag);
#pragma unroll
        for (int r = 0; r < US; ++r) {
            es[r] = as ? ne[r] : es[r];
            ee[r] = ae ? ne[r] : ee[r];
            wr[r] = accept ? nr[r] : wr[r];
            wi[r] = accept ? ni[r] : wi[r];
        }
        Gs = as ? nl : Gs;
        Ge = ae ? nl : Ge;
        Gp = accept ? np : Gp;
        const uint64_t bit = diag ? ((1ull << f.site) | (1ull << (f.site + N))) : (1ull << f.site);
        key ^= accept ? bit : 0ull;
        acc += accept ? 1u : 0u;
        f.site = site2;
        f.u = u2;
    };
    const int calls = a.burn + a.stored;
    int since = 0;
    for (int call = 0; call < calls; ++call) {
        // the factors from the configuration, so that rounding never accumulates over more than
        // kRatioRefresh proposals (or one call's)
        if (call == 0 || since + a.passes > kRatioRefresh) {
            since = 0;
            double ls = 1.0, le = 1.0, lp = 1.0;
#pragma unroll
            for (int r = 0; r < US; ++r) {
                const int h = hu[r] < 0 ? 0 : hu[r], q = au[r] < 0 ? 0 : au[r];
                es[r] = ee[r] = e0[r];
                wr[r] = w0[r];
                wi[r] = 0.0;
                for (int i = 0; i < N; ++i) {
                    const bool us = ((key >> i) & 1ull) != 0, ue = ((key >> (i + N)) & 1ull) != 0;
                    const double f = tl[i * nh + h].x;
                    const double2 p = tp[i * na + q];
                    es[r] *= us ? f : 1.0;
                    ee[r] *= ue ? f : 1.0;
                    // row and column side of the same site at +1: the phases cancel
                    const bool both = us && ue, one = us != ue;
                    const double pr = both && !diag ? p.x * p.x + p.y * p.y : (both || one ? p.x : 1.0);
                    const double pi = one ? (us ? p.y : -p.y) : 0.0;
                    const double t = wr[r] * pr - wi[r] * pi;
                    wi[r] = wr[r] * pi + wi[r] * pr;
                    wr[r] = t;
                }
                ls *= kl[r] + es[r];
                le *= kl[r] + ee[r];
                const double dr = kp[r] + wr[r];
                lp *= diag ? dr : dr * dr + wi[r] * wi[r];   // on the diagonal p ~ |rho|, z real
            }
            Gs = group_product<LPC>(ls);
            Ge = group_product<LPC>(le);
            Gp = group_product<LPC>(lp);
        }
        since += a.passes;
        int n = 0;
        for (; n + 2 <= a.passes; n += 2) {
            step(f0, f1);
            step(f1, f0);
        }
        if (n < a.passes) {
            step(f0, f1);
            const flip t = f0;
            f0 = f1;
            f1 = t;
        }
        if (call >= a.burn && live && gw == 0 && a.samples) {
            const int slice = a.slice0 + call - a.burn;
            a.samples[chain + (int64_t)slice * a.chains] = key;
        }
    }
    if (live && gw == 0) {
        if (a.chain_state) a.chain_state[chain] = key;
        if (a.compat_stale_last_slice && a.samples)
            a.samples[chain + (int64_t)(a.stored) * a.chains] = 0ull;   // defect D1: slice L stays at the fill
        if (a.accepted) atomicAdd(a.accepted, (unsigned long long)acc);
        if (a.chain_acc) a.chain_acc[chain] += (uint32_t)acc;   // one lane per chain: no race
    }
    return true;
}

template <int US, int ACT>
__global__ __launch_bounds__(256) void k_metropolis(samp_args a) {
    metropolis_body<float, US, ACT>(a, blockIdx.x);
}

// FP64 chains: by products where the weights' range allows it, else by sums of f
template <int LPC, int US, int ACT>
__device__ __forceinline__ void metropolis_f64(const samp_args& a, int bx) {
    if (a.diag ? metropolis_ratio_body<LPC, US, ACT, true>(a, bx) : metropolis_ratio_body<LPC, US, ACT, false>(a, bx)) return;
    __syncthreads();
    metropolis_body<double, US, ACT>(a, bx);
}
template <int LPC, int US, int ACT>
__global__ __launch_bounds__(256) void k_metropolis_f64(samp_args a) {
    metropolis_f64<LPC, US, ACT>(a, blockIdx.x);
}

// packed: the members' sampler launches in one grid (block records as in nq_pk_member)
template <typename T, int ACT>
__global__ __launch_bounds__(256) void k_metropolis_pk(const nq_pk_member* M, const uint2* blk) {
    const uint2 b = blk[blockIdx.x];
    const samp_args a = M[b.x & 0xffff].sa;
    const int bx = (int)(b.y & 0xffff);
    if constexpr (sizeof(T) == 8) {
        if (a.lpc == 8) metropolis_f64<8, 1, ACT>(a, bx);
        else if (a.lpc == 16) metropolis_f64<16, 1, ACT>(a, bx);
        else if (a.lpc == 32) metropolis_f64<32, 1, ACT>(a, bx);
        else metropolis_body<T, 1, ACT>(a, bx);   // fewer lanes: more chains than block records at 8
    } else {
        metropolis_body<T, 1, ACT>(a, bx);
    }
}

constexpr int kSampWaves = 4;   // wavefronts per workgroup (default)
constexpr int64_t kRepLanes = 1024 * 64;   // one wave per SIMD

int samp_waves(const samp_args& a) { return (a.waves == 1 || a.waves == 2 || a.waves == 4) ? a.waves : kSampWaves; }

int64_t samp_grid(const samp_args& a) {
    const int cpw = 64 / (a.lpc * a.rep);
    const int64_t waves = (a.chains + cpw - 1) / cpw;
    return (waves + samp_waves(a) - 1) / samp_waves(a);
}

// dynamic LDS: the parameters, or in FP64 the product tables in their place
size_t samp_lds(const ndm_dims& d, bool fp64) {
    const size_t par = (fp64 ? sizeof(double) : sizeof(float)) * (size_t)d.np;
    return fp64 ? std::max(par, ratio_lds_bytes(d)) : par;
}

template <int US>
hipError_t launch_f32(const samp_args& a, hipStream_t st) {
    const dim3 grid((unsigned)samp_grid(a)), blk(64 * samp_waves(a));
    const size_t lds = samp_lds(a.d, false);
    if (a.d.act == NQ_ACT_LOGCOSH)
        hipLaunchKernelGGL((k_metropolis<US, NQ_ACT_LOGCOSH>), grid, blk, lds, st, a);
    else
        hipLaunchKernelGGL((k_metropolis<US, NQ_ACT_SOFTPLUS>), grid, blk, lds, st, a);
    return hipGetLastError();
}

template <int LPC, int US>
hipError_t launch_f64(const samp_args& a, hipStream_t st) {
    const dim3 grid((unsigned)samp_grid(a)), blk(64 * samp_waves(a));
    const size_t lds = samp_lds(a.d, true);
    if (a.d.act == NQ_ACT_LOGCOSH)
        hipLaunchKernelGGL((k_metropolis_f64<LPC, US, NQ_ACT_LOGCOSH>), grid, blk, lds, st, a);
    else
        hipLaunchKernelGGL((k_metropolis_f64<LPC, US, NQ_ACT_SOFTPLUS>), grid, blk, lds, st, a);
    return hipGetLastError();
}

}  // namespace

// one unit of each kind per lane; at least 8 lanes in FP64 (its group width is a template argument)
int nq_sampler_lanes_per_chain(const ndm_dims& d, bool fp64) {
    const int m = d.nh > d.na ? d.nh : d.na;
    int l = fp64 ? 8 : 1;
    while (l < m && l < 64) l <<= 1;
    return l;
}

hipError_t nq_launch_metropolis(const samp_args& a0, bool fp64, hipStream_t st) {
    samp_args a = a0;
    const int m = a.d.nh > a.d.na ? a.d.nh : a.d.na;
    a.rep = 1;
    // FP64: while the chains leave SIMDs without a wave, copies of a group share a wave and with it
    // the draws (a wave's Philox pass then covers 64 proposals of one chain): 16 chains of 6 sites
    // 1.8 -> 1.2 ms per launch
    while (fp64 && a.lpc * a.rep < 64 && a.chains * a.lpc * a.rep * 2 <= kRepLanes) a.rep *= 2;
    // and with more than one wave per SIMD a lane takes several units instead, which shares the
    // proposal's overhead (draws, table index, acceptance) between them: 4096 chains of the 4x4 XYZ
    // network 0.95 ms at one unit per lane (2 waves per SIMD), 0.84 at two (1), 1.18 at four (1/2)
    while (fp64 && a.lpc > 8 && 4 * (a.lpc / 2) >= m && a.chains * a.lpc > kRepLanes) a.lpc /= 2;
    if (a.d.N > 32 || a.lpc < 1 || a.lpc > 64 || (a.lpc & (a.lpc - 1)) || m > 4 * a.lpc) return hipErrorInvalidValue;
    if (!fp64) return m > a.lpc ? hipErrorInvalidValue : launch_f32<1>(a, st);
    switch (10 * a.lpc + (m + a.lpc - 1) / a.lpc) {
        case 81: return launch_f64<8, 1>(a, st);
        case 82: return launch_f64<8, 2>(a, st);
        case 83: case 84: return launch_f64<8, 4>(a, st);
        case 161: return launch_f64<16, 1>(a, st);
        case 162: return launch_f64<16, 2>(a, st);
        case 163: case 164: return launch_f64<16, 4>(a, st);
        case 321: return launch_f64<32, 1>(a, st);
        case 322: return launch_f64<32, 2>(a, st);
        case 641: return launch_f64<64, 1>(a, st);
        default: return hipErrorInvalidValue;
    }
}

// packed launches: one lane group per chain covers every unit (lanes per
// chain >= max(nh, na), so one unit slot per lane); variant = fp64 | logcosh << 1
int nq_sampler_variant(const samp_args& a, bool fp64, int* threads, size_t* lds, int* grid) {
    const int m = a.d.nh > a.d.na ? a.d.nh : a.d.na;
    if (a.d.N > 32 || a.lpc < 1 || a.lpc > 64 || (a.lpc & (a.lpc - 1)) || m > a.lpc) return -1;
    const int64_t g = samp_grid(a);
    if (g > 0xffff) return -1;
    *threads = 64 * samp_waves(a);
    *lds = samp_lds(a.d, fp64);
    *grid = (int)g;
    return (fp64 ? 1 : 0) | (a.d.act == NQ_ACT_LOGCOSH ? 2 : 0);
}

hipError_t nq_pk_sampler(const nq_pk_member* M, const nq_pk_launch& L, hipStream_t st) {
    if (L.nblk <= 0) return hipSuccess;
    const dim3 g((unsigned)L.nblk), b((unsigned)L.threads);
    switch (L.variant) {
        case 0: hipLaunchKernelGGL((k_metropolis_pk<float, NQ_ACT_SOFTPLUS>), g, b, L.lds, st, M, L.blk); break;
        case 1: hipLaunchKernelGGL((k_metropolis_pk<double, NQ_ACT_SOFTPLUS>), g, b, L.lds, st, M, L.blk); break;
        case 2: hipLaunchKernelGGL((k_metropolis_pk<float, NQ_ACT_LOGCOSH>), g, b, L.lds, st, M, L.blk); break;
        case 3: hipLaunchKernelGGL((k_metropolis_pk<double, NQ_ACT_LOGCOSH>), g, b, L.lds, st, M, L.blk); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}
