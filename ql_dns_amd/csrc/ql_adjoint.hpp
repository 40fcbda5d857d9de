// ql_adjoint.hpp -- reverse-mode (adjoint) kernels of one RK3 substep of the
// MHD_FullQlin and MHD_BQlin quasilinear steps in FP64
// (Models/MHD_FullQlin.cpp:171-427, Models/MHD_BQlin.cpp:117-306, with the
// substep updates of Integrators/RK3CN_Elin.cpp:290-378 and
// Integrators/RK3CN.cpp:92-193).
//
// Gradients of a real loss L with respect to a complex value z are carried as
// G = dL/dRe z + i dL/dIm z, so dL = Re(conj(G) dz).  For z' = a z the
// reverse rule is G_z += conj(a) G_z'; for r = Re(a conj b) it is
// G_a += dL/dr b and G_b += dL/dr a.
//
// The transposes of the dealiased transforms are the other transform: the
// adjoint of "zero-pad nz -> NZ, unnormalised exp(+i) transform" is the
// unnormalised exp(-i) transform followed by truncation NZ -> nz, and vice
// versa, so the reverse pass reuses the forward transform code unchanged.
//
// One reverse substep (host sequence, ql_adjoint.hip):
//   k_adj_mf      one workgroup: z-profile adjoint of the substep reversed
//                 before into dL/dM and parameter gradient accumulation, then
//                 mean-field update and mean-field RHS in reverse, drive (EMF /
//                 stress) reverse down to dL/d(stress z-profiles) by an inverse
//                 transform;
//   k_adj_mode    per mode: recompute the forward lines and products, then
//                 reverse the update, the RHS assembly, the forward transforms,
//                 the mean-field x fluctuation products and the EMF / stress
//                 products, the inverse transforms and the base fields; per
//                 workgroup partial rows of dL/d(mean-field z-profiles) and of
//                 the parameter gradients;
//   k_reduce_cols column sum of those rows.
// The remap decision (MHD_FullQlin.cpp:470-472) is piecewise constant in q and
// enters as a fixed mask.
#pragma once
#include <type_traits>

#include "ql_mode.hpp"
#include "ql_noise.hpp"

namespace qlk {

// parameter-gradient slots (columns after the 8 z-profiles of a partial row)
enum { GP_Q = 0, GP_OMEGA = 1, GP_NU = 2, GP_ETA = 3, GP_B0Z = 4, NGP = 8 };

// d/dx of -|x|^p (neg_abs_pow)
__device__ __forceinline__ double neg_abs_pow_d(double x, int p)
{
    if (p == 0) return 0.0;
    const double a = fabs(x), sg = x < 0 ? -1.0 : (x > 0 ? 1.0 : 0.0);
    if (p == 1) return -sg;
    if (p == 2) return -2.0 * x;
    return -(double)p * pow_call(a, p - 1) * sg;
}

struct AdjModeArgs {
    const double2 *u_in;   // state at the substep start [nxy][4][nz]
    const double2 *u_out;  // state after the substep (after the remap at s = 3)
    double2 *gu;           // in: dL/du_out; out: dL/du_in
    double2 *gnp;          // in (s < 3): dL/dN_s via substep s+1; out (s > 1): dL/dN_{s-1}
    const double *kx0, *ky, *kzv;
    const double2 *tw;
    const double *mfz;     // z-profiles of the substep's mean fields [8][NZ]
    const double *gsums;   // dL/d(EMF / stress z-profiles) [4][NZ]
    double *gpart;         // [gridDim.x][8 NZ + NGP]
    Phys ph;
    int nxy, s, mode, do_remap, oinit;
    double rsf, remap_thr, fac;
    double linC, nlc1, nlc2;
    double ts, dtl, tso, dtlo, tnew;  // substep times (sub_times of the forward)
    // driving noise added after substep 3 (before the remap): its multipliers
    // depend on q through kx(t) at the step start t_step
    NoiseParams np;
    int noise;
    double t_step, dt_step;
};

// compact kz-slot lines ([line][LD]) as the first-pass source of an inverse
// transform (zero in the dealiased band) and the last-pass sink of a forward one
template <int NZ, int LD>
struct CompactIO {
    double2 *v;
    __device__ double2 operator()(int line, int g) const
    {
        using D = Dealias<NZ>;
        return D::kept(g) ? v[line * LD + D::slot(g)] : make_double2(0.0, 0.0);
    }
    __device__ void operator()(int line, int j, double2 x) const
    {
        using D = Dealias<NZ>;
        if (D::kept(j)) v[line * LD + D::slot(j)] = x;
    }
};

// inverse transform of NL compact lines in buf, in place (lines of LS slots)
template <int NZ, int NL, int LS, int LD>
__device__ __forceinline__ void adj_inv(double2 *buf, const double2 *tw)
{
    using PL = Plan2<NZ>;
    const PadIO<NZ, double2> pad{buf};
    fft_pass_io<NZ, NL, true, PL::R1, 1, true>(tw, CompactIO<NZ, LD>{buf}, pad);
    fft_pass_io<NZ, NL, true, PL::R2, PL::R1, true>(tw, pad, BufIO<LS, double2>{buf});
}
// forward transform of NL lines of LS slots in buf to compact lines, in place
template <int NZ, int NL, int LS, int LD>
__device__ __forceinline__ void adj_fwd(double2 *buf, const double2 *tw)
{
    using PL = Plan2<NZ>;
    const PadIO<NZ, double2> pad{buf};
    fft_pass_io<NZ, NL, false, PL::R1, 1, true>(tw, BufIO<LS, double2>{buf}, pad);
    fft_pass_io<NZ, NL, false, PL::R2, PL::R1, true>(tw, pad, CompactIO<NZ, LD>{buf});
}

// dL/dq through the step's driving noise (ql_noise.hpp) of one entry.  The
// noise is state independent; its ux and bx multipliers sqrt(nf lap2 / lapF)
// depend on q through lapF = -kx(t)^2 + lap2, d/dq = mult kx t ky / lapF (ky =
// 0 modes: none); the band mask is held fixed like the remap decision.  A
// call of its own: the generator's registers are not the mode kernel's
static __device__ __noinline__ double noise_q_gradient(NoiseParams np, double q, double tn, double dt,
                                                       double kx0, double ky, double kz2, int mode, int slot,
                                                       double2 gux, double2 gbx)
{
    const double kxn = rn_add(kx0, rn_mul(rn_mul(q, tn), ky));
    const double lap2n = rn_add(rn_mul(-ky, ky), kz2);
    const double lapF = rn_add(rn_mul(-kxn, kxn), lap2n);
    if (!(lapF > -np.hi2 && lapF < -np.lo2)) return 0.0;
    const double nf = rn_mul(dt, np.nfac);
    const double mu = sqrt(rn_mul(nf, lap2n) / lapF);
    double2 z[4];
    noise_normals(np.seed, tn, mode, slot, 0, z);
    noise_normals(np.seed, tn, mode, slot, 1, z + 2);
    double gz = 0.0;
    if (np.drive_u) gz += redot(z[0], gux);
    if (np.drive_b) gz += redot(z[2], gbx);
    return mu * kxn * (tn * ky) / lapF * np.sigma * gz;
}

// P = ModelFull (MHD_FullQlin) or ModelBQ (MHD_BQlin.cpp:117-306: 8 base
// lines, 5 product lines, By profiles only, no B0z terms, and the dz uz
// constant of the ky = 0 modes, whose gradient is summed over z per mode).
//
// A 256-thread workgroup takes MB = 256 / NZ modes at a time, as the forward
// workgroup kernel does: a thread owns one (mode, kz slot) in the spectral
// stages, whose state and gradients it keeps in registers, and one (mode, z)
// in the products.  Two line buffers in LDS (X lines, T lines: 52 KB at NZ =
// 128, two workgroups per CU) and the two-pass transforms in place in them.
// The recomputation transforms only the product lines the reverse reads: the
// momentum lines of MHD_FullQlin (the induction lines enter N linearly with
// constant factors) and the second line of MHD_BQlin.  Bound by the transforms
// (21 lines per mode, LDS and FP64 issue).  Against three radix-8 passes over
// unpadded lines with all 24 transforms and the products in two halves (rocprof,
// us): 64x64x128 RK3CN 132.8 -> 36.8, 32x32x64 RK3CN_Elin 19.8 -> 14.2.
template <int NZ, class P, int MODE>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(2))) void k_adj_mode(AdjModeArgs a)
{
    constexpr bool BQ = std::is_same<P, ModelBQ>::value;
    using D = Dealias<NZ>;
    constexpr int MB = NT / NZ, NZD = D::nz, NZDP = bank_stride(NZD), LS = bank_stride(NZ);
    constexpr int NIT = MB * NZD;       // (mode slot, kz slot) items
    constexpr int NLX = P::NLINE * MB;  // 6 (8) lines per mode
    constexpr int NLG = P::NOUT * MB;   // 6 (5) gradient lines per mode
    constexpr int L0 = BQ ? 1 : 0;      // the product lines the reverse reads: L0 .. L0 + NRD - 1
    constexpr int NRD = BQ ? 1 : 3;
    constexpr int XS = Plan2Size<NZ, NLX, LS>::SLOTS, TS = Plan2Size<NZ, NLG, LS>::SLOTS;
    static_assert(MB * NZ == NT && NIT <= NT, "one item per thread");
    static_assert(NLX * NZDP <= XS && NLG * NZDP <= TS, "compact lines fit the line buffers");
    __shared__ double2 bufX[XS];  // bases, X lines, dL/dX lines, their spectra
    __shared__ double2 bufT[TS];  // products, T, dL/dT, dL/dP lines
    __shared__ double2 tw[NZ];
    __shared__ double smfz[P::NMFZ * NZ];  // mean-field profiles [profile][z]
    __shared__ double sgs[4 * NZ];         // dL/d(EMF / stress sums) [slot][z]
    __shared__ double skx[MB], sky[MB];
    __shared__ int sok[MB];
    __shared__ double2 sdz[MB];               // ModelBQ: fac ux at kz = 0 of a ky = 0 mode
    constexpr int SEG = NZ < 64 ? NZ : 64;    // lanes of a wavefront on one mode's z points
    __shared__ double2 sgdz[BQ ? NT / SEG : 1];  // ModelBQ: partial sums of that value's gradient
    const int tid = threadIdx.x;
    const Phys ph = a.ph;
    const double q = ph.q, Om = ph.omega, B0z = ph.B0z;
    // d op / d x of a dissipation operator coef op(x), x = -kx^2 - ky^2 + kz2: -|x|^p
    // for MHD_FullQlin, x itself for MHD_BQlin
    const auto opd = [&](double x) { return BQ ? 1.0 : neg_abs_pow_d(x, ph.vo2); };
    const double qt = to_sgpr(rn_mul(q, a.ts)), qdtl = to_sgpr(rn_mul(q, a.dtl));
    const double qt_old = to_sgpr(rn_mul(q, a.tso)), qdtl_old = to_sgpr(rn_mul(q, a.dtlo));
    const double remap_qt = to_sgpr(rn_mul(q, a.tnew));
    const bool remap_now = a.s == 3 && a.do_remap;

    // the thread's items, fixed for the whole kernel
    const bool has_it = tid < NIT;
    const int imb = tid / NZD, im = tid - imb * NZD;
    const int zmb = tid / NZ, zz = tid - zmb * NZ;
    const double kz = has_it ? a.kzv[im] : 0.0, kz2 = -(kz * kz);
    for (int k = tid; k < P::NMFZ * NZ; k += NT) smfz[k] = a.mfz[k];
    for (int k = tid; k < 4 * NZ; k += NT) sgs[k] = a.gsums[k];
    if (tid < NZ) tw[tid] = a.tw[tid];

    // per-thread gradient accumulators: parameters and z-profile rows
    double gq = 0, gom = 0, gnu = 0, geta = 0, gb0 = 0;
    double accm[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) accm[c] = 0.0;

    const int ngroups = (a.nxy + MB - 1) / MB;
    for (int g = blockIdx.x; g < ngroups; g += gridDim.x) {
        // A, B: the item's state row and wavenumbers, the bases (forward
        // recomputation)
        const int i = (has_it && g * MB + imb < a.nxy) ? g * MB + imb : -1;
        const size_t off = (size_t)(i < 0 ? 0 : i) * 4 * NZD + im;
        const double kx0 = i >= 0 ? a.kx0[i] : 0.0, ky = i >= 0 ? a.ky[i] : 0.0;
        const double kx = i >= 0 ? rn_add(kx0, rn_mul(qt, ky)) : 0.0;
        const bool zero = (ky == 0.0 && im == 0);
        const double lap2 = zero ? 0.0 : (-ky * ky + kz2);
        const double ilap2 = zero ? 1.0 : 1.0 / lap2;
        if (has_it) {
            double2 u[4];
#pragma unroll
            for (int f = 0; f < 4; ++f) u[f] = i >= 0 ? a.u_in[off + f * NZD] : make_double2(0.0, 0.0);
            P::bases(u[0], u[1], u[2], u[3], kx, ky, kz, ilap2, a.fac, bufX + imb * NZDP + im, MB * NZDP);
            if (im == 0) {
                skx[imb] = kx;
                sky[imb] = ky;
                sok[imb] = i >= 0;
                sdz[imb] = (BQ && i >= 0 && ky == 0.0) ? cscale(a.fac, u[0]) : make_double2(0.0, 0.0);
            }
        }
        __syncthreads();
        adj_inv<NZ, NLX, LS, NZDP>(bufX, tw);

        // D, E: the product lines the reverse reads and their transforms
        const double zkx = skx[zmb], zky = sky[zmb];
        const bool zok = sok[zmb] != 0;
        double2 *X = bufX + zmb * LS + zz;  // line l at X[l * MB * LS]
        double2 *Y = bufT + zmb * LS + zz;
        {
            double2 prod[3];
            double racc[2], mf[P::NMFZ];
#pragma unroll
            for (int c = 0; c < P::NMFZ; ++c) mf[c] = smfz[c * NZ + zz];
            P::products(0, X, MB * LS, mf, zkx, zky, imul(zkx, sdz[zmb]), prod, racc);
#pragma unroll
            for (int c = 0; c < NRD; ++c) Y[c * MB * LS] = prod[L0 + c];
        }
        __syncthreads();
        adj_fwd<NZ, NRD * MB, LS, NZDP>(bufT, tw);

        // F: substep update and RHS assembly in reverse, per (mode, kz slot)
        double2 *GT = bufT + imb * NZDP + im;  // T (line c at c * MB * NZDP), then dL/dT
        if (has_it && i < 0)
            for (int o = 0; o < P::NOUT; ++o) GT[o * MB * NZDP] = make_double2(0.0, 0.0);
        if (i >= 0) {
            double2 u[4];
#pragma unroll
            for (int f = 0; f < 4; ++f) u[f] = a.u_in[off + f * NZD];
            const double2 ux = u[0], ze = u[1], bx = u[2], et = u[3];
            double2 gout[4], GN[4], gdir[4];
            const bool hit = remap_now && remap_hit(remap_qt, a.remap_thr, kx0, ky);
#pragma unroll
            for (int f = 0; f < 4; ++f) gout[f] = hit ? make_double2(0.0, 0.0) : a.gu[off + f * NZD];
            if (a.noise && a.s == 3 && !hit && a.np.sigma != 0.0 && ky != 0.0)
                gq += noise_q_gradient(a.np, q, a.t_step, a.dt_step, kx0, ky, kz2, i, im, gout[0], gout[2]);
            const double kxn = kx + qdtl * ky;
            const double xn = (-kxn * kxn - ky * ky) + kz2;
            double xo = 0.0, dxo_dq = 0.0, kxo_e = 0.0;
            const double kxo = rn_add(kx0, rn_mul(qt_old, ky));
            if constexpr (MODE == MODE_CN) {
                if (a.oinit) {
                    xo = -kxo * kxo + lap2;
                    kxo_e = kxo;
                    dxo_dq = a.tso * ky;
                } else {
                    kxo_e = kxo + qdtl_old * ky;
                    xo = (-kxo_e * kxo_e - ky * ky) + kz2;
                    dxo_dq = (a.tso + a.dtlo) * ky;
                }
            }
            // the operators and their derivatives, which the pairs share
            const double opn = P::op(xn, ph), dpn = opd(xn);
            const double opo = MODE == MODE_CN ? P::op(xo, ph) : 0.0, dpo = MODE == MODE_CN ? opd(xo) : 0.0;
#pragma unroll
            for (int pr = 0; pr < 2; ++pr) {
                const double coef = pr == 0 ? ph.nu : ph.eta;
                const double Ln = P::lin(pr, opn, ph);
                double gLn = 0.0, gLo = 0.0;
                // factors of the update and of the two right-hand sides in it
                double e, d = 1.0;
                if constexpr (MODE == MODE_ELIN) {
                    e = exp(a.linC * Ln);
                } else {
                    const double Lo = P::lin(pr, opo, ph);
                    d = 1.0 / (1.0 - a.linC * Ln);
                    e = (1 + a.linC * Lo) * d;
                }
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int f = 2 * pr + h;
                    const double2 go = gout[f];
                    const double2 gin = (a.s < 3) ? a.gnp[off + f * NZD] : make_double2(0.0, 0.0);
                    const double2 uo = a.u_out[off + f * NZD];
                    if constexpr (MODE == MODE_ELIN) {
                        const double2 mu = cscale(e, go);
                        GN[f] = cadd(cscale(a.nlc1, mu), gin);
                        if (a.s > 1) a.gnp[off + f * NZD] = cscale(a.nlc2, mu);
                        gdir[f] = mu;
                        gLn += a.linC * redot(uo, go);
                    } else {
                        GN[f] = cadd(cscale(a.nlc1 * d, go), gin);
                        if (a.s > 1) a.gnp[off + f * NZD] = cscale(a.nlc2 * d, go);
                        gdir[f] = cscale(e, go);
                        gLn += a.linC * d * redot(uo, go);
                        gLo += a.linC * d * redot(u[f], go);
                    }
                }
                // L = coef * op(x): coefficient and kx(t) = kx0 + q t ky dependence
                const double gc = gLn * opn + (MODE == MODE_CN ? gLo * opo : 0.0);
                if (pr == 0) gnu += gc;
                else geta += gc;
                gq += gLn * coef * dpn * (-2.0 * kxn) * ((a.ts + a.dtl) * ky);
                if (MODE == MODE_CN) gq += gLo * coef * dpo * (-2.0 * kxo_e) * dxo_dq;
            }
            const double ilapF = (i == 0 && im == 0) ? 1.0 : 1.0 / (-kx * kx + lap2);
            if constexpr (!BQ) {
                // RHS assembly in reverse (MHD_FullQlin.cpp:283-285, :303-305)
                const double2 T1 = GT[0], T2 = GT[MB * NZDP], T3 = GT[2 * MB * NZDP];
                double gkx = 0.0;
                // N_ux = ilapF s + i B0z kz bx - T1,  s = 2 kx ky q ux + i 2 Om kz ze - kx^2 T1 - kx ky T2 - kx kz T3
                double2 s = cscale(2.0 * kx * ky * q, ux);
                s = cadd(s, imul(2.0 * Om * kz, ze));
                s = csub(s, cscale(kx * kx, T1));
                s = csub(s, cscale(kx * ky, T2));
                s = csub(s, cscale(kx * kz, T3));
                const double2 Gs = cscale(ilapF, GN[0]);
                double2 GT0 = csub(cscale(-kx * kx, Gs), GN[0]);
                double2 GT1 = cscale(-kx * ky, Gs);
                double2 GT2 = cscale(-kx * kz, Gs);
                gdir[0] = cadd(gdir[0], cscale(2.0 * kx * ky * q, Gs));
                gdir[1] = cadd(gdir[1], imul(-2.0 * Om * kz, Gs));
                gdir[2] = cadd(gdir[2], imul(-B0z * kz, GN[0]));
                {
                    double2 dsk = cscale(2.0 * ky * q, ux);
                    dsk = csub(dsk, cscale(2.0 * kx, T1));
                    dsk = csub(dsk, cscale(ky, T2));
                    dsk = csub(dsk, cscale(kz, T3));
                    gkx += redot(dsk, Gs);
                }
                if (!(i == 0 && im == 0)) gkx += redot(s, GN[0]) * 2.0 * kx * ilapF * ilapF;
                gq += redot(cscale(2.0 * kx * ky, ux), Gs);
                gom += redot(imul(2.0 * kz, ze), Gs);
                gb0 += redot(imul(kz, bx), GN[0]);
                // N_ze = i (q - 2 Om) kz ux + i B0z kz et - i kz T2 + i ky T3
                gdir[0] = cadd(gdir[0], imul(-(q - 2.0 * Om) * kz, GN[1]));
                gdir[3] = cadd(gdir[3], imul(-B0z * kz, GN[1]));
                GT1 = cadd(GT1, imul(kz, GN[1]));
                GT2 = cadd(GT2, imul(-ky, GN[1]));
                gq += redot(imul(kz, ux), GN[1]);
                gom += redot(imul(-2.0 * kz, ux), GN[1]);
                gb0 += redot(imul(kz, et), GN[1]);
                // N_bx = i B0z kz ux - T4
                gdir[0] = cadd(gdir[0], imul(-B0z * kz, GN[2]));
                gb0 += redot(imul(kz, ux), GN[2]);
                // N_et = -i q kz bx + i B0z kz ze - i kz T5 + i ky T6
                gdir[2] = cadd(gdir[2], imul(q * kz, GN[3]));
                gdir[1] = cadd(gdir[1], imul(-B0z * kz, GN[3]));
                gq += redot(imul(-kz, bx), GN[3]);
                gb0 += redot(imul(kz, ze), GN[3]);
                gq += gkx * (a.ts * ky);
                GT[0] = GT0;
                GT[MB * NZDP] = GT1;
                GT[2 * MB * NZDP] = GT2;
                GT[3 * MB * NZDP] = cscale(-1.0, GN[2]);
                GT[4 * MB * NZDP] = imul(kz, GN[3]);
                GT[5 * MB * NZDP] = imul(-ky, GN[3]);
            } else {
                // MHD_BQlin.cpp:160-162, :177-178, :185, :200-201 in reverse:
                // N_ux = T1 + ilapF (s + T2), s = 2 kx ky q ux + i 2 Om kz ze;
                // N_ze = T4 + i (q - 2 Om) kz ux; N_bx = T3; N_et = T5 - i q kz bx
                const double2 T2 = GT[0];  // the only line transformed
                double gkx = 0.0;
                const double2 s = cadd(cscale(2.0 * kx * ky * q, ux), imul(2.0 * Om * kz, ze));
                const double2 Gs = cscale(ilapF, GN[0]);
                gdir[0] = cadd(gdir[0], cscale(2.0 * kx * ky * q, Gs));
                gdir[1] = cadd(gdir[1], imul(-2.0 * Om * kz, Gs));
                gkx += redot(cscale(2.0 * ky * q, ux), Gs);
                if (!(i == 0 && im == 0)) gkx += redot(cadd(s, T2), GN[0]) * 2.0 * kx * ilapF * ilapF;
                gq += redot(cscale(2.0 * kx * ky, ux), Gs);
                gom += redot(imul(2.0 * kz, ze), Gs);
                gdir[0] = cadd(gdir[0], imul(-(q - 2.0 * Om) * kz, GN[1]));
                gq += redot(imul(kz, ux), GN[1]);
                gom += redot(imul(-2.0 * kz, ux), GN[1]);
                gdir[2] = cadd(gdir[2], imul(q * kz, GN[3]));
                gq += redot(imul(-kz, bx), GN[3]);
                gq += gkx * (a.ts * ky);
                GT[0] = GN[0];
                GT[MB * NZDP] = Gs;
                GT[2 * MB * NZDP] = GN[2];
                GT[3 * MB * NZDP] = GN[1];
                GT[4 * MB * NZDP] = GN[3];
            }
            // the direct terms wait in the gradient itself for J
#pragma unroll
            for (int f = 0; f < 4; ++f) a.gu[off + f * NZD] = gdir[f];
        }
        __syncthreads();

        // G: adjoint of the forward transforms = padded inverse transforms
        adj_inv<NZ, NLG, LS, NZDP>(bufT, tw);

        // H: products and EMF / stress terms in reverse, per (mode, z); the X
        // lines of the thread's z point become their gradients
        double2 gdz = make_double2(0.0, 0.0);
        if (!zok) {
#pragma unroll
            for (int l = 0; l < P::NLINE; ++l) X[l * MB * LS] = make_double2(0.0, 0.0);
        } else if constexpr (BQ) {
            // MHD_BQlin products (MHD_BQlin.cpp:153-201, :219-240) in reverse;
            // X lines ux ze bx et uy uz by bz, P lines: By i ky bx,
            // dzBy 2 kx ky bz, By i ky ux, (zeta), (eta)
            const double2 ux = X[0], ze = X[MB * LS], bx = X[2 * MB * LS], et = X[3 * MB * LS];
            const double2 uy = X[4 * MB * LS], uz = X[5 * MB * LS], by = X[6 * MB * LS], bz = X[7 * MB * LS];
            const double2 G0 = Y[0], G1 = Y[MB * LS], G2 = Y[2 * MB * LS], G3 = Y[3 * MB * LS], G4 = Y[4 * MB * LS];
            const double By = smfz[zz], dzBy = smfz[NZ + zz], dzdzBy = smfz[2 * NZ + zz];
            const double ftfac = (zky == 0.0 ? 1.0 : 2.0) * a.rsf;
            const double g0 = ftfac * sgs[zz], g1 = ftfac * sgs[NZ + zz];  // EMF x, EMF y
            double gkx = 0.0;
            // ux, ze, uy, uz; dz uz = -i kx ux - i ky uy + dzc enters the
            // eta product as dzBy (-2 dz uz - i kx ux)
            const double2 dzuz = cadd(cadd(imul(-zkx, ux), imul(-zky, uy)), imul(zkx, sdz[zmb]));
            const double2 t2 = csub(cscale(-2.0, dzuz), imul(zkx, ux));
            X[0] = cadd(cadd(imul(-zky * By, G2), imul(-zkx * dzBy, G4)), cscale(g0, bz));
            X[MB * LS] = imul(-zky * By, G4);
            X[4 * MB * LS] = cadd(imul(-2.0 * zky * dzBy, G4), cscale(g1, bz));
            X[5 * MB * LS] = csub(cscale(-dzdzBy, G4), cadd(cscale(g0, bx), cscale(g1, by)));
            gdz = cscale(-2.0 * dzBy, G4);
            accm[0] += redot(imul(zky, ux), G2) + redot(imul(zky, ze), G4);
            accm[1] += redot(t2, G4);
            accm[2] -= redot(uz, G4);
            gkx += redot(imul(dzBy, ux), G4);
            // bx, et, by, bz
            X[2 * MB * LS] = csub(cadd(imul(-zky * By, G0), imul(zkx * dzBy, G3)), cscale(g0, uz));
            X[3 * MB * LS] = imul(-zky * By, G3);
            X[6 * MB * LS] = cscale(-g1, uz);
            X[7 * MB * LS] = cadd(cadd(cscale(2.0 * zkx * zky * dzBy, G1), cscale(dzdzBy, G3)),
                                  cadd(cscale(g0, ux), cscale(g1, uy)));
            accm[0] += redot(imul(zky, bx), G0) + redot(imul(zky, et), G3);
            accm[1] += redot(cscale(2.0 * zkx * zky, bz), G1) + redot(imul(-zkx, bx), G3);
            accm[2] += redot(bz, G3);
            gkx += redot(cscale(2.0 * zky * dzBy, bz), G1) + redot(imul(-dzBy, bx), G3);
            gq += gkx * (a.ts * zky);
        } else {
            const double2 u0 = X[0], u1 = X[MB * LS], u2 = X[2 * MB * LS];
            const double2 b0 = X[3 * MB * LS], b1 = X[4 * MB * LS], b2 = X[5 * MB * LS];
            const double2 G0 = Y[0], G1 = Y[MB * LS], G2 = Y[2 * MB * LS];
            const double2 G3 = Y[3 * MB * LS], G4 = Y[4 * MB * LS], G5 = Y[5 * MB * LS];
            const double *mf = smfz + zz;
            const double MBx = mf[0], dzMBx = mf[NZ], MBy = mf[2 * NZ], dzMBy = mf[3 * NZ];
            const double MUx = mf[4 * NZ], dzMUx = mf[5 * NZ], MUy = mf[6 * NZ], dzMUy = mf[7 * NZ];
            const double aU = zkx * MUx + zky * MUy, aB = zkx * MBx + zky * MBy;
            const double ftfac = (zky == 0.0 ? 1.0 : 2.0) * a.rsf;
            const double g0 = ftfac * sgs[zz], g1 = ftfac * sgs[NZ + zz], g2 = ftfac * sgs[2 * NZ + zz],
                         g3 = ftfac * sgs[3 * NZ + zz];
            // u0 (0), u1 (1), u2 (2)
            double2 Gu0 = cadd(imul(-aU, G0), imul(aB, G3));
            double2 Gu1 = cadd(imul(-aU, G1), imul(aB, G4));
            double2 Gu2 = cadd(cadd(cscale(dzMUx, G0), cscale(dzMUy, G1)), imul(-aU, G2));
            Gu2 = cadd(Gu2, cadd(cadd(cscale(dzMBx, G3), cscale(dzMBy, G4)), imul(aB, G5)));
            // EMF x, y (slots 0, 1) and stresses (slots 2, 3:
            // -Re(uz conj(ux)), -Re(uz conj(uy)) before their z-derivative)
            Gu0 = cadd(Gu0, cscale(g0, b2));
            Gu2 = csub(Gu2, cadd(cscale(g0, b0), cscale(g1, b1)));
            Gu1 = cadd(Gu1, cscale(g1, b2));
            Gu0 = csub(Gu0, cscale(g2, u2));
            Gu1 = csub(Gu1, cscale(g3, u2));
            Gu2 = csub(Gu2, cadd(cscale(g2, u0), cscale(g3, u1)));
            X[0] = Gu0;
            X[MB * LS] = Gu1;
            X[2 * MB * LS] = Gu2;
            // b0 (0), b1 (1), b2 (2)
            double2 Gb0 = cadd(imul(aB, G0), imul(-aU, G3));
            double2 Gb1 = cadd(imul(aB, G1), imul(-aU, G4));
            double2 Gb2 = cadd(cadd(cscale(-dzMBx, G0), cscale(-dzMBy, G1)), imul(aB, G2));
            Gb2 = cadd(Gb2, cadd(cadd(cscale(-dzMUx, G3), cscale(-dzMUy, G4)), imul(-aU, G5)));
            Gb2 = cadd(Gb2, cadd(cscale(g0, u0), cscale(g1, u1)));
            Gb0 = csub(Gb0, cscale(g0, u2));
            Gb1 = csub(Gb1, cscale(g1, u2));
            // stresses: +Re(bz conj(bx)), +Re(bz conj(by))
            Gb0 = cadd(Gb0, cscale(g2, b2));
            Gb1 = cadd(Gb1, cscale(g3, b2));
            Gb2 = cadd(Gb2, cadd(cscale(g2, b0), cscale(g3, b1)));
            X[3 * MB * LS] = Gb0;
            X[4 * MB * LS] = Gb1;
            X[5 * MB * LS] = Gb2;
            // mean-field profile and kx gradients: the momentum products, then
            // the induction products
            double gaU = redot(imul(1.0, u0), G0) + redot(imul(1.0, u1), G1) + redot(imul(1.0, u2), G2);
            double gaB = redot(imul(-1.0, b0), G0) + redot(imul(-1.0, b1), G1) + redot(imul(-1.0, b2), G2);
            gaU += redot(imul(1.0, b0), G3) + redot(imul(1.0, b1), G4) + redot(imul(1.0, b2), G5);
            gaB += redot(imul(-1.0, u0), G3) + redot(imul(-1.0, u1), G4) + redot(imul(-1.0, u2), G5);
            accm[0] += zkx * gaB;
            accm[1] += redot(u2, G3) - redot(b2, G0);  // dz MBx
            accm[2] += zky * gaB;
            accm[3] += redot(u2, G4) - redot(b2, G1);  // dz MBy
            accm[4] += zkx * gaU;
            accm[5] += redot(u2, G0) - redot(b2, G3);  // dz MUx
            accm[6] += zky * gaU;
            accm[7] += redot(u2, G1) - redot(b2, G4);  // dz MUy
            gq += (MUx * gaU + MBx * gaB) * (a.ts * zky);
        }
        if constexpr (BQ) {
            // the dz uz constant's gradient summed over z: within a wavefront
            // here, over a mode's wavefronts by its reader in J
#pragma unroll
            for (int o = SEG / 2; o > 0; o >>= 1)
                gdz = cadd(gdz, make_double2(__shfl_xor(gdz.x, o), __shfl_xor(gdz.y, o)));
            if (tid % SEG == 0) sgdz[tid / SEG] = gdz;
        }
        __syncthreads();

        // I: adjoint of the padded inverse transforms = truncated forward transforms
        adj_fwd<NZ, NLX, LS, NZDP>(bufX, tw);

        // J: base fields in reverse; total dL/du_in
        if (i >= 0) {
            const double2 *GL = bufX + imb * NZDP + im;  // line l at GL[l * MB * NZDP]
            const double f = a.fac;
            const double2 ux = a.u_in[off], bx = a.u_in[off + 2 * NZD];
            // the y, z bases: uy = (ky kx ux + i kz ze) ilap2, uz = (kx kz ux - i ky ze)
            // ilap2 (and b likewise), all bases times fac
            const double2 GBx = GL[0], GBy = GL[(BQ ? 4 : 1) * MB * NZDP], GBz = GL[(BQ ? 5 : 2) * MB * NZDP];
            const double2 Gbx_ = GL[(BQ ? 2 : 3) * MB * NZDP], Gby_ = GL[(BQ ? 6 : 4) * MB * NZDP],
                          Gbz_ = GL[(BQ ? 7 : 5) * MB * NZDP];
            const double2 G1z = BQ ? GL[MB * NZDP] : make_double2(0.0, 0.0);      // the zeta base
            const double2 G3e = BQ ? GL[3 * MB * NZDP] : make_double2(0.0, 0.0);  // the eta base
            double2 Gux = cscale(f, cadd(GBx, cadd(cscale(ky * kx * ilap2, GBy), cscale(kx * kz * ilap2, GBz))));
            double2 Gze = cadd(imul(-kz * ilap2, GBy), imul(ky * ilap2, GBz));
            const double2 Gbx = cscale(f, cadd(Gbx_, cadd(cscale(ky * kx * ilap2, Gby_), cscale(kx * kz * ilap2, Gbz_))));
            double2 Get = cadd(imul(-kz * ilap2, Gby_), imul(ky * ilap2, Gbz_));
            if constexpr (BQ) {
                Gze = cadd(G1z, Gze);
                Get = cadd(G3e, Get);
            }
            Gze = cscale(f, Gze);
            Get = cscale(f, Get);
            double gkx = f * (redot(cscale(ky * ilap2, ux), GBy) + redot(cscale(kz * ilap2, ux), GBz) +
                              redot(cscale(ky * ilap2, bx), Gby_) + redot(cscale(kz * ilap2, bx), Gbz_));
            if (BQ && zero) {
                // dzc = i kx (fac ux at kz = 0) of a ky = 0 mode
                double2 Gd = sgdz[imb * (NZ / SEG)];
#pragma unroll
                for (int w = 1; w < NZ / SEG; ++w) Gd = cadd(Gd, sgdz[imb * (NZ / SEG) + w]);
                Gux = cadd(Gux, imul(-kx * f, Gd));
                gkx += redot(imul(1.0, sdz[imb]), Gd);
            }
            gq += gkx * (a.ts * ky);
            const double2 total[4] = {Gux, Gze, Gbx, Get};
#pragma unroll
            for (int fl = 0; fl < 4; ++fl) a.gu[off + fl * NZD] = cadd(a.gu[off + fl * NZD], total[fl]);
        }
        __syncthreads();
    }

    // partial row of this workgroup: the z-profile gradients summed over the
    // mode slots, then the parameter gradients over the threads, both in a
    // fixed order
    double *red = reinterpret_cast<double *>(bufX);
    static_assert((8 * NT + 5 * (NT / 64)) * sizeof(double) <= sizeof(bufX), "reduction fits the X lines");
    double *row = a.gpart + (size_t)blockIdx.x * (8 * NZ + NGP);
#pragma unroll
    for (int c = 0; c < 8; ++c) red[(zmb * 8 + c) * NZ + zz] = accm[c];
    double gp[5] = {gq, gom, gnu, geta, gb0};
#pragma unroll
    for (int c = 0; c < 5; ++c) {
        const double t = wave_sum(gp[c]);
        if (tid % 64 == 0) red[8 * NT + c * (NT / 64) + tid / 64] = t;
    }
    __syncthreads();
    for (int k = tid; k < 8 * NZ; k += NT) {
        double s = 0.0;
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) s += red[mb * 8 * NZ + k];
        row[k] = s;
    }
    if (tid < NGP) {
        double s = 0.0;
        if (tid < 5)
            for (int w = 0; w < NT / 64; ++w) s += red[8 * NT + tid * (NT / 64) + w];
        row[8 * NZ + tid] = s;
    }
}

// ---------------------------------------------------------------------------
// mean fields in reverse, one workgroup between the mode kernels of two
// reverse substeps: first the z-profile adjoint of the substep just reversed
// (rows), then the update, RHS and drive of the next one (s).  Two two-pass
// transforms between separate LDS regions; latency-bound, like k_meanfield (32x32x64:
// 5.5 us, 8.7 for the two launches it replaces).
// ---------------------------------------------------------------------------
struct AdjMFArgs {
    // z-profile part (rows null: none): adds the profiles' gradient to gM and
    // the substep's parameter gradients (rows' and gpar's) to gpar_total
    const double *rows;  // reduced partial rows [8 NZ + NGP]
    double *gpar_total;  // [NGP]
    double fac;
    // update part (s = 0: none)
    double2 *gM;           // in: dL/dM_out; out: dL/dM_in without the z-profile path
    double2 *gnmp;         // in (s < 3): dL/dNM_s; out (s > 1): dL/dNM_{s-1}
    const double2 *M_in, *M_out;
    const double *kzv;
    const double2 *tw;
    double *gsums;         // out: dL/d(EMF / stress z-profiles) [4][NZ]
    double *gpar;          // parameter-gradient partials [NGP] of the substep's mean fields
    Phys ph;
    int mode, s;
    double linC, nlc1, nlc2;
};

// MODEL 0: MHD_FullQlin (Bx, By, Ux, Uy); 1: MHD_BQlin (Bx, By: N_Bx = EMF x,
// N_By = -q Bx + EMF y, both with eta kz^2, MHD_BQlin.cpp:274-280).  The
// z-profiles are mfz_l = Re(inverse(pad(c_l M))) with c = fac (l even) or
// i fac kz (l odd) (MHD_FullQlin.cpp:180-198); MHD_BQlin's are By, dz By, dz^2
// By with c = fac, i fac kz, -fac kz^2 (MHD_BQlin.cpp:122-127), Bx has none.
template <int NZ, int MODEL>
__global__ __launch_bounds__(NT) void k_adj_mf(AdjMFArgs a)
{
    using D = Dealias<NZ>;
    using PL = Plan2<NZ>;
    constexpr int NZD = D::nz, HALF = D::half;
    constexpr int NM = MODEL == 0 ? 4 : 2, NP = MODEL == 0 ? 8 : 3;
    constexpr int KW = (NM * NZD + NT - 1) / NT;
    __shared__ double2 padb[8 * PadIO<NZ, double2>::LP];
    __shared__ double2 line[8 * NZ];
    __shared__ double2 tw[NZ];
    __shared__ double skz[NZD];
    __shared__ double2 sGN[4 * NZD], sM[4 * NZD];
    __shared__ double red[5][NT / 64];
    const int tid = threadIdx.x;
    const Phys ph = a.ph;
    const PadIO<NZ, double2> pad{padb};
    const BufIO<NZ, double2> lines{line};
    // loads of both parts first, so that they are in flight together
    double2 g[KW], gin[KW], Mo[KW], Mi[KW];
#pragma unroll
    for (int w = 0; w < KW; ++w) {
        const int k = tid + w * NT;
        const bool ok = k < NM * NZD, up = ok && a.s > 0;
        g[w] = ok ? a.gM[k] : make_double2(0.0, 0.0);
        gin[w] = (up && a.s < 3) ? a.gnmp[k] : make_double2(0.0, 0.0);
        Mo[w] = up ? a.M_out[k] : make_double2(0.0, 0.0);
        Mi[w] = up ? a.M_in[k] : make_double2(0.0, 0.0);
    }
    if (tid < NZ) tw[tid] = a.tw[tid];
    if (tid < NZD) skz[tid] = a.kzv[tid];
    if (a.rows && tid < NGP) a.gpar_total[tid] += a.gpar[tid] + a.rows[8 * NZ + tid];
    __syncthreads();
    if (a.rows) {
        const double *R = a.rows;
        const auto ld = [R](int l, int j) { return make_double2(R[l * NZ + j], 0.0); };
        fft_pass_io<NZ, NP, false, PL::R1, 1, false>(tw, ld, pad);
        fft_pass_io<NZ, NP, false, PL::R2, PL::R1, false>(tw, pad, lines);
#pragma unroll
        for (int w = 0; w < KW; ++w) {
            const int k = tid + w * NT;
            if (k >= NM * NZD) continue;
            const int f = k / NZD, m = k % NZD;
            const double kz = skz[m];
            const int j = D::pad(m);
            if (MODEL == 0) {
                g[w] = cadd(g[w], cadd(cscale(a.fac, line[(2 * f) * NZ + j]),
                                       imul(-a.fac * kz, line[(2 * f + 1) * NZ + j])));
            } else if (f == 1) {
                double2 G = cadd(cscale(a.fac, line[j]), imul(-a.fac * kz, line[NZ + j]));
                g[w] = cadd(g[w], cadd(G, cscale(-a.fac * kz * kz, line[2 * NZ + j])));
            }
        }
    }
    if (a.s == 0) {
#pragma unroll
        for (int w = 0; w < KW; ++w)
            if (tid + w * NT < NM * NZD) a.gM[tid + w * NT] = g[w];
        return;
    }
    double gq = 0, gom = 0, gnu = 0, geta = 0, gb0 = 0;
    double2 dir[KW];
    // update in reverse (RK3CN_Elin.cpp:109-112 / RK3CN.cpp:112-115)
#pragma unroll
    for (int w = 0; w < KW; ++w) {
        const int k = tid + w * NT;
        dir[w] = make_double2(0.0, 0.0);
        if (k >= NM * NZD) continue;
        const int f = k / NZD, m = k % NZD;
        const double kz2 = -(skz[m] * skz[m]);
        const double coef = f < 2 ? ph.eta : ph.nu;
        const double L = ph.quasilinear ? coef * kz2 : 0.0;
        double2 GN;
        double gL;
        if (a.mode == MODE_ELIN) {
            const double2 mu = cscale(exp(a.linC * L), g[w]);
            GN = cadd(cscale(a.nlc1, mu), gin[w]);
            if (a.s > 1) a.gnmp[k] = cscale(a.nlc2, mu);
            dir[w] = mu;
            gL = a.linC * redot(Mo[w], g[w]);
        } else {
            const double d = 1.0 / (1.0 - a.linC * L);
            GN = cadd(cscale(a.nlc1 * d, g[w]), gin[w]);
            if (a.s > 1) a.gnmp[k] = cscale(a.nlc2 * d, g[w]);
            dir[w] = cscale((1 + a.linC * L) * d, g[w]);
            gL = a.linC * d * (redot(Mi[w], g[w]) + redot(Mo[w], g[w]));
        }
        if (ph.quasilinear) {
            if (f < 2) geta += gL * kz2;
            else gnu += gL * kz2;
        }
        sGN[k] = ph.quasilinear ? GN : make_double2(0.0, 0.0);
        sM[k] = Mi[w];
    }
    __syncthreads();
    // mean-field RHS in reverse (MHD_FullQlin.cpp:411-423)
#pragma unroll
    for (int w = 0; w < KW; ++w) {
        const int k = tid + w * NT;
        if (k >= NM * NZD) continue;
        const int f = k / NZD, m = k % NZD;
        const double kz = skz[m];
        double2 G = dir[w];
        if constexpr (MODEL == 1) {
            if (f == 0) {
                G = cadd(G, cscale(-ph.q, sGN[NZD + m]));
                gq += redot(cscale(-1.0, sM[m]), sGN[NZD + m]);
            }
            a.gM[k] = G;
        } else {
            const double2 N0 = sGN[m], N1 = sGN[NZD + m], N2 = sGN[2 * NZD + m], N3 = sGN[3 * NZD + m];
            if (f == 0) G = cadd(G, cadd(cscale(-ph.q, N1), imul(-ph.B0z * kz, N2)));
            else if (f == 1) G = cadd(G, imul(-ph.B0z * kz, N3));
            else if (f == 2) G = cadd(G, cadd(imul(-ph.B0z * kz, N0), cscale(ph.q - 2.0 * ph.omega, N3)));
            else G = cadd(G, cadd(imul(-ph.B0z * kz, N1), cscale(2.0 * ph.omega, N2)));
            a.gM[k] = G;
            if (f == 0) {
                const double2 M0 = sM[m], M1 = sM[NZD + m], M2 = sM[2 * NZD + m], M3 = sM[3 * NZD + m];
                gq += redot(cscale(-1.0, M0), N1) + redot(M2, N3);
                gom += redot(cscale(2.0, M3), N2) + redot(cscale(-2.0, M2), N3);
                gb0 += redot(imul(kz, M2), N0) + redot(imul(kz, M3), N1) + redot(imul(kz, M0), N2) +
                       redot(imul(kz, M1), N3);
            }
        }
    }
    // drive in reverse: Hermitian fill and x i kz of every line (the EMF,
    // MHD_FullQlin.cpp:326-336, and the stresses before their z-derivative),
    // then the forward transform's adjoint (an inverse transform) of the
    // real stress profiles
    const auto src = [&](int f, int n) {
        double2 v = make_double2(0.0, 0.0);
        if (n < HALF) {
            const double c = skz[n];
            v = imul(-c, sGN[f * NZD + n]);
            const int mm = 2 * HALF - 1 - n;  // slot filled with conj of this one
            if (n >= 1 && mm < NZD) {
                double2 d1 = sGN[f * NZD + mm];
                d1.y = -d1.y;
                v = cadd(v, imul(-c, d1));
            }
        }
        return v;
    };
    double *gs = a.gsums;
    const auto out = [gs](int l, int i, double2 v) { gs[l * NZ + i] = v.x; };
    fft_pass_io<NZ, NM, true, PL::R1, 1, false>(tw, src, pad);
    fft_pass_io<NZ, NM, true, PL::R2, PL::R1, false>(tw, pad, out);
    const double gp[5] = {gq, gom, gnu, geta, gb0};
#pragma unroll
    for (int c = 0; c < 5; ++c) {
        const double t = wave_sum(gp[c]);
        if (tid % 64 == 0) red[c][tid / 64] = t;
    }
    __syncthreads();
    if (tid < NGP) {
        double s = 0.0;
        if (tid < 5)
            for (int w = 0; w < NT / 64; ++w) s += red[tid][w];
        a.gpar[tid] = s;
    }
}

}  // namespace qlk
