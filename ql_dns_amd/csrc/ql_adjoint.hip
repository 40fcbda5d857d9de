// ql_adjoint.hip -- adjoint (reverse-mode gradient) of n steps of the QL main
// loop (main.cpp:108-123: Step, t += dt, ShearingBox_Remap) for one
// MHD_FullQlin or MHD_BQlin run in FP64, with checkpointed recomputation.
//
// ql_adjoint_forward runs the steps exactly as ql_steps does (the same kernels
// and launch shape, so the same bits) and stores the state every `every`
// steps.  ql_adjoint_backward walks the segments backwards: it restores a
// checkpoint, recomputes the segment's substeps eagerly, each writing its state,
// mean fields and profiles to buffers of its own (3 every + 1 states), then runs
// the reverse substeps (ql_adjoint.hpp) from the last to the first.  It returns dL/d(state at the
// start of the forward) and dL/d(q, omega, nu, eta, B0z) for the caller's
// dL/d(final state); the context is left at the final state of the forward.
#include <algorithm>
#include <cstdio>
#include <cstring>

#include "ql_adjoint.hpp"
#include "ql_runtime.hpp"
#include "ql_state_out.hpp"

namespace qlh {

// Everything one context's gradients need.  It stays with the context, so that
// a loop of gradients allocates once; a forward with other steps or spacing
// gives back what no longer fits (adj_fit).
struct AdjState {
    bool valid = false;  // a forward has completed
    int nsteps = 0, every = 0, nseg = 0;
    bool noise = false;  // the forward was driven
    // checkpoints at segment starts (index nseg: the final state); with
    // variable steps also the step taken last and the profile maxima the next
    // step's dt comes from
    struct Ck {
        double2 *u = nullptr, *mf = nullptr;
        double *kx0 = nullptr, *pm = nullptr;
        double t = 0.0, t_prev = 0.0, dt_last = 0.0;
        int old_init = 0;
    };
    std::vector<Ck> ck;
    double2 *drive = nullptr;  // of the forward's last right-hand side (no segment reads them)
    double t_init = 0.0;
    // substep states, mean fields and profiles of one segment; with driving
    // noise also each step's state after substep 3 before the noise and the
    // remap
    double2 *st_u = nullptr, *st_mf = nullptr, *st_pre = nullptr;
    double *st_kx0 = nullptr, *st_mfz = nullptr;
    // adjoint buffers
    double2 *gu = nullptr, *gnp = nullptr, *gM = nullptr, *gnmp = nullptr;
    double *gsums = nullptr, *gpart = nullptr, *grows = nullptr, *gpar_mf = nullptr, *gpar = nullptr;
};

// The buffers outlive a call that fails, so each of the three kinds (a
// checkpoint, the segment's, the adjoint's) is there as a whole or not at all:
// its first pointer tells
namespace {
void free_ck(AdjState::Ck &c) { dfree(c.u), dfree(c.mf), dfree(c.kx0), dfree(c.pm); }
void free_segment(AdjState *A)
{
    dfree(A->st_u), dfree(A->st_mf), dfree(A->st_kx0), dfree(A->st_pre), dfree(A->st_mfz);
}
void free_adjoint(AdjState *A)
{
    dfree(A->gu), dfree(A->gnp), dfree(A->gM), dfree(A->gnmp);
    dfree(A->gsums), dfree(A->gpart), dfree(A->grows), dfree(A->gpar_mf), dfree(A->gpar);
}
}  // namespace

void adj_release(Batch &b)
{
    AdjState *A = b.adj;
    if (!A) return;
    for (auto &c : A->ck) free_ck(c);
    dfree(A->drive);
    free_segment(A);
    free_adjoint(A);
    delete A;
    b.adj = nullptr;
}

namespace {

// workgroups of the reverse mode kernel, at most: two per CU
constexpr int ADJ_GMAX = 512;

int check_adjoint(const Batch &b, const char *who)
{
    if (b.runs.size() != 1) return fail(QL_ERR_UNSUPPORTED, "%s: the adjoint is for single-run contexts", who);
    if (b.model != QL_MODEL_MHD_FULLQLIN && b.model != QL_MODEL_MHD_BQLIN && !b.hd)
        return fail(QL_ERR_UNSUPPORTED, "%s: the adjoint is implemented for MHD_FullQlin, MHD_BQlin and HD_fullU", who);
    if (b.precision != QL_PREC_FP64) return fail(QL_ERR_UNSUPPORTED, "%s: the adjoint runs in FP64 only", who);
    return QL_OK;
}

// a checkpoint's buffers: all of them or none
int alloc_ck(AdjState::Ck &c, const Group &g, size_t nl, size_t nm)
{
    const int rc = [&]() -> int {
        QL_RC(dalloc_queued(&c.u, nl));
        QL_RC(dalloc_queued(&c.mf, nm));
        QL_RC(dalloc_queued(&c.kx0, g.modes));
        QL_RC(dalloc_queued(&c.pm, (size_t)qlk::PM_STRIDE));
        return dwait();
    }();
    if (rc != QL_OK) free_ck(c);
    return rc;
}

// checkpoint k of the forward
int save_ck(Batch &b, int k, double t)
{
    AdjState *A = b.adj;
    AdjState::Ck &c = A->ck[k];
    Group &g = b.groups[0];
    const size_t nl = (size_t)g.modes * 4 * g.nz, nm = (size_t)b.nMF * g.nz;
    if (!c.u) {
        int rc = alloc_ck(c, g, nl, nm);
        if (rc != QL_OK && (A->st_u || A->gu)) {
            // what an earlier backward left makes way
            QL_HIP(hipStreamSynchronize(b.s));
            free_segment(A);
            free_adjoint(A);
            rc = alloc_ck(c, g, nl, nm);
        }
        QL_RC(rc);
    }
    QL_HIP(hipMemcpyAsync(c.u, g.u, sizeof(double2) * nl, hipMemcpyDeviceToDevice, b.s));
    QL_HIP(hipMemcpyAsync(c.mf, g.mf, sizeof(double2) * nm, hipMemcpyDeviceToDevice, b.s));
    QL_HIP(hipMemcpyAsync(c.kx0, g.kx0, sizeof(double) * g.modes, hipMemcpyDeviceToDevice, b.s));
    QL_HIP(hipMemcpyAsync(c.pm, g.pm, sizeof(double) * qlk::PM_STRIDE, hipMemcpyDeviceToDevice, b.s));
    c.t = t;
    c.t_prev = b.t_prev;
    c.dt_last = b.dt_last;
    c.old_init = b.old_init;
    return QL_OK;
}

// the state, step record and clock history of a checkpoint, the state into u, mf
// and the profiles mfz
int load_ck(Batch &b, const AdjState::Ck &c, double2 *u, double2 *mf, double *mfz)
{
    Group &g = b.groups[0];
    const size_t nl = (size_t)g.modes * 4 * g.nz, nm = (size_t)b.nMF * g.nz;
    QL_HIP(hipMemcpyAsync(u, c.u, sizeof(double2) * nl, hipMemcpyDeviceToDevice, b.s));
    QL_HIP(hipMemcpyAsync(mf, c.mf, sizeof(double2) * nm, hipMemcpyDeviceToDevice, b.s));
    QL_HIP(hipMemcpyAsync(g.kx0, c.kx0, sizeof(double) * g.modes, hipMemcpyDeviceToDevice, b.s));
    QL_HIP(hipMemcpyAsync(g.pm, c.pm, sizeof(double) * qlk::PM_STRIDE, hipMemcpyDeviceToDevice, b.s));
    b.t_prev = c.t_prev;
    b.dt_last = c.dt_last;
    b.old_init = c.old_init;
    qlk::MFArgs m = mf_args(b, g);
    m.mf = mf;
    m.mfz = mfz;
    m.rec = 0;  // the record is the checkpoint's: HD_fullU's holds the drives of its last rhs
    launch_profiles(b, g, m, b.s);
    QL_HIP(hipGetLastError());
    return QL_OK;
}

// substep times of the forward (sub_times in ql_kernels.hpp, same roundings);
// dt_last, the step before (equal to dt with fixed steps), places the RK3CN
// "old" operator of substep 1
struct HostTimes {
    double ts, dtl, tso, dtlo, tnew;
    int oinit;
};
HostTimes host_times(double t, double t_prev, int old_init, double t_init, double dt, double dt_last, int s)
{
    HostTimes r{};
    const double dtP1 = dt * P1, dtP2 = dt * P2;
    const double dtl1 = dt * P1, dtl2 = dt * (P2 - P1), dtl3 = dt * (1.0 - P2);
    const double dtP2o = dt_last * P2, dtl3o = dt_last * (1.0 - P2);
    r.tnew = t + dt;
    if (s == 1) {
        r.ts = t;
        r.dtl = dtl1;
        r.oinit = old_init;
        r.tso = old_init ? t_init : t_prev + dtP2o;
        r.dtlo = old_init ? 0.0 : dtl3o;
    } else if (s == 2) {
        r.ts = t + dtP1;
        r.dtl = dtl2;
        r.tso = t;
        r.dtlo = dtl1;
    } else {
        r.ts = t + dtP2;
        r.dtl = dtl3;
        r.tso = t + dtP1;
        r.dtlo = dtl2;
    }
    return r;
}

template <int NZ, int MODEL>
void launch_adj_mode_nz(const qlk::AdjModeArgs &am, int W, double *grows, hipStream_t st)
{
    using P = typename std::conditional<MODEL == 0, qlk::ModelFull, qlk::ModelBQ>::type;
    if (am.mode == qlk::MODE_CN) qlk::k_adj_mode<NZ, P, qlk::MODE_CN><<<W, qlk::NT, 0, st>>>(am);
    else qlk::k_adj_mode<NZ, P, qlk::MODE_ELIN><<<W, qlk::NT, 0, st>>>(am);
    const int ncols = 8 * NZ + qlk::NGP;
    qlk::k_reduce_cols<<<dim3((ncols + qlk::RED_CW - 1) / qlk::RED_CW, 1), qlk::NT, 0, st>>>(am.gpart, nullptr, W, ncols, grows);
}

template <int MODEL>
void launch_adj_mode_m(int NZ, const qlk::AdjModeArgs &am, int W, double *grows, hipStream_t st)
{
    switch (NZ) {
    case 32: launch_adj_mode_nz<32, MODEL>(am, W, grows, st); break;
    case 64: launch_adj_mode_nz<64, MODEL>(am, W, grows, st); break;
    case 128: launch_adj_mode_nz<128, MODEL>(am, W, grows, st); break;
    default: launch_adj_mode_nz<256, MODEL>(am, W, grows, st); break;
    }
}

// the reverse mode kernel and the column sums of its partial rows
int launch_adj_mode(int NZ, int model, const qlk::AdjModeArgs &am, int W, double *grows, hipStream_t st)
{
    if (model == QL_MODEL_MHD_BQLIN) launch_adj_mode_m<1>(NZ, am, W, grows, st);
    else launch_adj_mode_m<0>(NZ, am, W, grows, st);
    QL_HIP(hipGetLastError());
    return QL_OK;
}

template <int NZ>
void launch_adj_mf_nz(int model, const qlk::AdjMFArgs &a, hipStream_t st)
{
    if (model == QL_MODEL_MHD_BQLIN) qlk::k_adj_mf<NZ, 1><<<1, qlk::NT, 0, st>>>(a);
    else qlk::k_adj_mf<NZ, 0><<<1, qlk::NT, 0, st>>>(a);
}

int launch_adj_mf(int NZ, int model, const qlk::AdjMFArgs &a, hipStream_t st)
{
    switch (NZ) {
    case 32: launch_adj_mf_nz<32>(model, a, st); break;
    case 64: launch_adj_mf_nz<64>(model, a, st); break;
    case 128: launch_adj_mf_nz<128>(model, a, st); break;
    default: launch_adj_mf_nz<256>(model, a, st); break;
    }
    QL_HIP(hipGetLastError());
    return QL_OK;
}

// The context's AdjState for a forward of nsteps with checkpoints every `every`
// steps: buffers of an earlier forward are kept where they fit and given back
// where they do not
int adj_fit(Batch &b, int nsteps, int every, bool noise)
{
    if (!b.adj) b.adj = new AdjState();
    AdjState *A = b.adj;
    A->valid = false;
    if (A->every != every || A->noise != noise) {
        QL_HIP(hipStreamSynchronize(b.s));
        free_segment(A);
    }
    A->nsteps = nsteps;
    A->every = every;
    A->nseg = (nsteps + every - 1) / every;
    A->noise = noise;
    if ((int)A->ck.size() > A->nseg + 1) {
        QL_HIP(hipStreamSynchronize(b.s));
        for (size_t k = A->nseg + 1; k < A->ck.size(); ++k) free_ck(A->ck[k]);
    }
    A->ck.resize(A->nseg + 1);
    return QL_OK;
}

// one segment's states, mean fields and profiles: all of them or none
int alloc_segment(AdjState *A, const Group &g, size_t nl, size_t nm)
{
    const size_t K = A->every;
    const int rc = [&]() -> int {
        QL_RC(dalloc_queued(&A->st_u, nl * (3 * K + 1)));
        QL_RC(dalloc_queued(&A->st_mf, nm * (3 * K + 1)));
        QL_RC(dalloc_queued(&A->st_kx0, (size_t)g.modes * K));
        // zeroed: MHD_BQlin writes 3 of the 8 profile lines
        QL_RC(dalloc_queued(&A->st_mfz, (size_t)8 * g.NZ * (3 * K + 1)));
        if (g.noise) QL_RC(dalloc_queued(&A->st_pre, nl * K));
        return dwait();
    }();
    if (rc != QL_OK) free_segment(A);
    return rc;
}

// the adjoint state, its sums and W partial rows: all of them or none
int alloc_adjoint(AdjState *A, const Group &g, size_t nl, size_t nm, int W)
{
    const size_t ncols = 8 * g.NZ + qlk::NGP;
    const int rc = [&]() -> int {
        QL_RC(dalloc_queued(&A->gu, nl));
        QL_RC(dalloc_queued(&A->gnp, nl));
        QL_RC(dalloc_queued(&A->gM, nm));
        QL_RC(dalloc_queued(&A->gnmp, nm));
        QL_RC(dalloc_queued(&A->gsums, (size_t)4 * g.NZ));  // zeroed: MHD_BQlin fills 2 of the 4 lines
        QL_RC(dalloc_queued(&A->gpart, (size_t)W * ncols));
        QL_RC(dalloc_queued(&A->grows, ncols));
        QL_RC(dalloc_queued(&A->gpar_mf, (size_t)qlk::NGP));
        QL_RC(dalloc_queued(&A->gpar, (size_t)qlk::NGP));
        return dwait();
    }();
    if (rc != QL_OK) free_adjoint(A);
    return rc;
}

int adjoint_forward(Batch &b, int nsteps, int every, double *t_inout)
{
    QL_RC(check_adjoint(b, "ql_adjoint_forward"));
    if (nsteps < 1 || every < 1) return fail(QL_ERR_ARG, "ql_adjoint_forward: nsteps=%d, every=%d", nsteps, every);
    QL_RC(adj_fit(b, nsteps, every, b.groups[0].noise));
    AdjState *A = b.adj;
    A->t_init = b.t_init;
    double t = *t_inout;
    for (int sg = 0; sg < A->nseg; ++sg) {
        QL_RC(save_ck(b, sg, t));
        const int n = std::min(every, nsteps - sg * every);
        QL_RC(run_steps(b, n, &t));
    }
    QL_RC(save_ck(b, A->nseg, t));
    const Group &g = b.groups[0];
    const size_t nm = (size_t)b.nMF * g.nz;
    if (!A->drive) QL_RC(dalloc(&A->drive, nm));
    QL_HIP(hipMemcpyAsync(A->drive, g.drive, sizeof(double2) * nm, hipMemcpyDeviceToDevice, b.s));
    QL_HIP(hipStreamSynchronize(b.s));
    A->valid = true;
    *t_inout = t;
    return QL_OK;
}

int adjoint_backward(Batch &b, const double *g_lin, const double *g_mf, double *g_lin0, double *g_mf0,
                     double *g_par)
{
    QL_RC(check_adjoint(b, "ql_adjoint_backward"));
    AdjState *A = b.adj;
    if (!A || !A->valid) return fail(QL_ERR_STATE, "ql_adjoint_backward: no ql_adjoint_forward on this context");
    if (A->noise != b.groups[0].noise)
        return fail(QL_ERR_STATE, "ql_adjoint_backward: the driving noise changed since ql_adjoint_forward");
    Group &g = b.groups[0];
    const RunInfo &r = b.runs[0];
    const int NZ = g.NZ, nz = g.nz, nxy = r.nxy, K = A->every;
    const size_t nl = (size_t)nxy * 4 * nz, nm = (size_t)b.nMF * nz;
    const int MB = qlk::NT / NZ;  // modes per pass of the reverse mode kernel
    const int W = std::min((nxy + MB - 1) / MB, ADJ_GMAX);
    if (!A->st_u) QL_RC(alloc_segment(A, g, nl, nm));
    if (!A->gu) QL_RC(alloc_adjoint(A, g, nl, nm, W));
    // HD_fullU runs the MHD_FullQlin kernels with b = B = 0 on the internal
    // four-field layout: its caller's (ux, zeta) and (Ux, Uy) gradients sit at
    // fields 0, 1 and mean-field slots 2, 3, the others are zero
    std::vector<double2> hl, hm;
    if (b.hd) {
        hl.assign(nl, make_double2(0.0, 0.0));
        hm.assign(nm, make_double2(0.0, 0.0));
        if (g_lin)
            for (int i = 0; i < nxy; ++i)
                std::memcpy(&hl[(size_t)i * 4 * nz], g_lin + (size_t)i * 2 * nz * 2, sizeof(double2) * 2 * nz);
        if (g_mf) std::memcpy(&hm[(size_t)2 * nz], g_mf, sizeof(double2) * 2 * nz);
        QL_HIP(hipMemcpy(A->gu, hl.data(), sizeof(double2) * nl, hipMemcpyHostToDevice));
        QL_HIP(hipMemcpy(A->gM, hm.data(), sizeof(double2) * nm, hipMemcpyHostToDevice));
    } else {
        if (g_lin) QL_HIP(hipMemcpyAsync(A->gu, g_lin, sizeof(double2) * nl, hipMemcpyHostToDevice, b.s));
        else QL_HIP(hipMemsetAsync(A->gu, 0, sizeof(double2) * nl, b.s));
        if (g_mf) QL_HIP(hipMemcpyAsync(A->gM, g_mf, sizeof(double2) * nm, hipMemcpyHostToDevice, b.s));
        else QL_HIP(hipMemsetAsync(A->gM, 0, sizeof(double2) * nm, b.s));
    }
    QL_HIP(hipMemsetAsync(A->gnp, 0, sizeof(double2) * nl, b.s));
    QL_HIP(hipMemsetAsync(A->gnmp, 0, sizeof(double2) * nm, b.s));
    QL_HIP(hipMemsetAsync(A->gpar, 0, sizeof(double) * qlk::NGP, b.s));

    const bool cn = (b.integrator == QL_INT_RK3CN);
    // the clock advances on the device through a segment; variable steps and
    // driven ones need the host's times step by step
    const bool stepwise = b.vdt || g.noise;
    bool have_rows = false;  // a reverse substep's sums wait for their z-profile adjoint
    qlk::AdjMFArgs aa{};
    aa.gpar_total = A->gpar;
    aa.fac = 1.0 / NZ;
    aa.gM = A->gM;
    aa.gnmp = A->gnmp;
    aa.kzv = g.kzv;
    aa.tw = g.tw;
    aa.gsums = A->gsums;
    aa.gpar = A->gpar_mf;
    aa.ph = g.h_rp[0].ph;
    aa.mode = cn ? qlk::MODE_CN : qlk::MODE_ELIN;
    for (int sg = A->nseg - 1; sg >= 0; --sg) {
        const int n = std::min(K, A->nsteps - sg * K);
        // recompute the segment, every substep into the next slot
        QL_RC(load_ck(b, A->ck[sg], A->st_u, A->st_mf, A->st_mfz));
        double t = A->ck[sg].t;
        std::vector<double> st_t(n), st_tp(n), st_dt(n), st_dtl(n);
        std::vector<int> st_oi(n);
        for (int k = 0; k < n; ++k) {
            st_t[k] = t;
            st_tp[k] = b.t_prev;
            st_oi[k] = b.old_init;
            QL_HIP(hipMemcpyAsync(A->st_kx0 + (size_t)k * nxy, g.kx0, sizeof(double) * nxy, hipMemcpyDeviceToDevice,
                                  b.s));
            if (k == 0 || stepwise) QL_RC(set_clock(b, t));
            // with variable steps the device chose the step from the profile
            // maxima, as in the forward (ql_step); the reverse takes it as given
            double dt = b.dt;
            if (b.vdt) {
                qlk::Clock ck{};
                QL_RC(read_clock(b, &ck));
                dt = ck.dt;
            }
            st_dt[k] = dt;
            st_dtl[k] = b.vdt ? b.dt_last : dt;
            for (int s = 1; s <= 3; ++s) {
                const size_t j = (size_t)3 * k + s;
                const SubBuffers bf{A->st_u + (j - 1) * nl, A->st_mf + (j - 1) * nm, A->st_u + j * nl,
                                    A->st_mf + j * nm, A->st_mfz + (j - 1) * 8 * NZ, A->st_mfz + j * 8 * NZ};
                // with noise the step's remap follows the noise (main.cpp:111-123)
                QL_RC(enqueue_substep(b, g, s, s == 3 && !g.noise, !stepwise, b.s, &bf));
                if (s == 3 && g.noise) {
                    QL_HIP(hipMemcpyAsync(A->st_pre + (size_t)k * nl, A->st_u + j * nl, sizeof(double2) * nl,
                                          hipMemcpyDeviceToDevice, b.s));
                    QL_RC(launch_noise(g, A->st_u + j * nl, false, t, dt, true, r.p.remap != 0, b.s));
                }
            }
            b.t_prev = t;
            b.dt_last = dt;
            b.old_init = 0;
            t = t + dt;
        }
        // reverse substeps
        for (int k = n - 1; k >= 0; --k) {
            for (int s = 3; s >= 1; --s) {
                const size_t jin = (size_t)3 * k + s - 1, jout = jin + 1;
                const double dt = st_dt[k];
                const HostTimes ht = host_times(st_t[k], st_tp[k], st_oi[k], A->t_init, dt, st_dtl[k], s);
                double lc, nlc1, nlc2 = 0.0;
                if (s == 1) {
                    lc = cn ? dt / 2 * (A0) : dt * (A0);
                    nlc1 = A0 * dt;
                } else if (s == 2) {
                    lc = cn ? dt / 2 * (A1 + B1) : dt * (A1 + B1);
                    nlc1 = A1 * dt;
                    nlc2 = B1 * dt;
                } else {
                    lc = cn ? dt / 2 * (A2 + B2) : dt * (A2 + B2);
                    nlc1 = A2 * dt;
                    nlc2 = B2 * dt;
                }
                // the substep reversed before: its z-profiles; this one: its
                // mean fields
                aa.rows = have_rows ? A->grows : nullptr;
                aa.M_in = A->st_mf + jin * nm;
                aa.M_out = A->st_mf + jout * nm;
                aa.s = s;
                aa.linC = lc;
                aa.nlc1 = nlc1;
                aa.nlc2 = nlc2;
                QL_RC(launch_adj_mf(NZ, b.model, aa, b.s));

                qlk::AdjModeArgs am{};
                am.u_in = A->st_u + jin * nl;
                // the substep's own output: before the step's noise at s = 3
                am.u_out = (s == 3 && g.noise) ? A->st_pre + (size_t)k * nl : A->st_u + jout * nl;
                am.gu = A->gu;
                am.gnp = A->gnp;
                am.kx0 = A->st_kx0 + (size_t)k * nxy;
                am.ky = g.ky;
                am.kzv = g.kzv;
                am.tw = g.tw;
                am.mfz = A->st_mfz + jin * 8 * NZ;
                am.gsums = A->gsums;
                am.gpart = A->gpart;
                am.ph = g.h_rp[0].ph;
                am.nxy = nxy;
                am.s = s;
                am.mode = aa.mode;
                am.do_remap = r.p.remap;
                am.oinit = ht.oinit;
                am.rsf = r.rsf;
                am.remap_thr = r.remap_thr;
                am.fac = 1.0 / NZ;
                am.linC = lc;
                am.nlc1 = nlc1;
                am.nlc2 = nlc2;
                am.ts = ht.ts;
                am.dtl = ht.dtl;
                am.tso = ht.tso;
                am.dtlo = ht.dtlo;
                am.tnew = ht.tnew;
                am.noise = g.noise ? 1 : 0;
                if (g.noise) am.np = g.h_np[0];
                am.t_step = st_t[k];
                am.dt_step = dt;
                QL_RC(launch_adj_mode(NZ, b.model, am, W, A->grows, b.s));
                have_rows = true;
            }
        }
    }
    aa.rows = have_rows ? A->grows : nullptr;
    aa.s = 0;
    QL_RC(launch_adj_mf(NZ, b.model, aa, b.s));
    // leave the context at the forward's final state
    QL_RC(load_ck(b, A->ck[A->nseg], g.u, g.mf, g.mfz));
    QL_HIP(hipMemcpyAsync(g.drive, A->drive, sizeof(double2) * nm, hipMemcpyDeviceToDevice, b.s));
    double gp[qlk::NGP];
    QL_RC(state_out(*b.out, b.s, A->gu, nxy, ext_nlin(b) * nz, 4 * nz, g_lin0, A->gM + (size_t)ext_mf0(b) * nz,
                    ext_nmf(b) * nz, g_mf0, A->gpar, qlk::NGP, gp));
    if (b.hd) gp[3] = gp[4] = 0.0;  // HD_fullU has no eta and no B0z
    if (b.model == QL_MODEL_MHD_BQLIN) {
        // MHD_BQlin rotates at 2 q / 3 whatever omega is (MHD_BQlin.cpp:19): the
        // kernels' rotation gradient belongs to q
        gp[0] += 2.0 / 3.0 * gp[1];
        gp[1] = 0.0;
    }
    if (g_par)
        for (int c = 0; c < 5; ++c) g_par[c] = gp[c];
    return QL_OK;
}

}  // namespace
}  // namespace qlh

using namespace qlh;

extern "C" {

int ql_adjoint_forward(ql_ctx *c, int nsteps, int every, double *t_inout)
{
    if (!c || !t_inout) return fail(QL_ERR_ARG, "ql_adjoint_forward: null argument");
    return adjoint_forward(c->bt.b, nsteps, every, t_inout);
}

int ql_adjoint_backward(ql_ctx *c, const double *g_lin, const double *g_mf, double *g_lin0, double *g_mf0,
                        double g_par[5])
{
    if (!c) return fail(QL_ERR_ARG, "ql_adjoint_backward: null context");
    return adjoint_backward(c->bt.b, g_lin, g_mf, g_lin0, g_mf0, g_par);
}

}  // extern "C"
