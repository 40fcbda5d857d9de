// ql_mode_wave.hpp -- the per-(kx,ky) substep kernel of MHD_FullQlin, MHD_BQlin
// and HD_fullU (through its velocity-only policy, ModelHD) with one wavefront
// per mode (Models/MHD_FullQlin.cpp:171-427, Models/MHD_BQlin.cpp:117-284,
// Models/HD_fullU.cpp:145-309 and the
// substep updates of Integrators/RK3CN_Elin.cpp:290-378,
// Integrators/RK3CN.cpp:92-193).
//
// Same stages as mode_body (ql_mode.hpp) -- bases, inverse transforms,
// products and EMF / stress sums, forward transforms, RHS and update -- but a
// wavefront takes a whole mode in a private LDS region, so the stages are
// ordered by wavefront-local fences instead of workgroup barriers and the
// wavefronts of a workgroup run independently; the other wavefronts of a SIMD
// hide a wavefront's memory and LDS latency.  The workgroup (NW wavefronts)
// shares the twiddle, wavenumber and profile tables and reduces its
// wavefronts' EMF / stress sums into one partial row at the end.  Every
// transform pass reads and writes the wavefront's buffer: it loads all its
// inputs before its first store, and a fence separates the two.  FP64 at NZ =
// 128 and 256 keeps the z lines in registers between the passes (RowPlan).
#pragma once
#include "ql_mode.hpp"

namespace qlk {

// Orders the LDS accesses of one wavefront: its LDS instructions execute in
// issue order, so waiting for the outstanding ones and keeping the compiler
// from moving memory accesses across is enough for its lanes to see each
// other's stores.  Global memory counters are not waited for.
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0); vmcnt, expcnt unchanged
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

constexpr int WAVE = 64;

// fft_pass_io for the 64 lanes of one wavefront
template <int NZ, int NL, bool INV, int R, int NS, class C, class Ld, class St>
__device__ __forceinline__ void wave_pass(int lane, const C *tw, const Ld &ld, const St &st)
{
    constexpr int M = NZ / R;
    constexpr int TOT = NL * M;
    constexpr int IT = (TOT + WAVE - 1) / WAVE;
    C v[IT][R];
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        const int item = lane + it * WAVE;
        if (TOT % WAVE == 0 || item < TOT) {
            const int line = item / M, j = item % M;
#pragma unroll
            for (int r = 0; r < R; ++r) v[it][r] = ld(line, j + r * M);
        }
    }
    wave_sync();
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        if (it > 0) __builtin_amdgcn_sched_barrier(0);  // one butterfly at a time (registers)
        const int item = lane + it * WAVE;
        if (TOT % WAVE == 0 || item < TOT) {
            const int line = item / M, j = item % M;
            const int k = j % NS;
            if constexpr (NS > 1) {
#pragma unroll
                for (int r = 1; r < R; ++r) {
                    C w = tw[k * r * (NZ / (NS * R))];
                    if (INV) w.y = -w.y;
                    v[it][r] = cmul(v[it][r], w);
                }
            }
            if constexpr (R == 16) {
                dft16<INV>(v[it]);
            } else if constexpr (R == 8) {
                dft8<INV>(v[it]);
            } else if constexpr (R == 4) {
                dft4<INV>(v[it][0], v[it][1], v[it][2], v[it][3]);
            } else {
                const C a = v[it][0], b = v[it][1];
                v[it][0] = cadd(a, b);
                v[it][1] = csub(a, b);
            }
#pragma unroll
            for (int r = 0; r < R; ++r) st(line, (j - k) * R + k + r * NS, v[it][r]);
        }
    }
    wave_sync();
}

// Two-way exchanges between the 16-lane rows of a wavefront (v_permlane32_swap,
// v_permlane16_swap): x and y as the columns of a 2 x 2 matrix whose rows are
// the wavefront's halves (its even and odd rows) are transposed
__device__ __forceinline__ void swap_halves(unsigned &x, unsigned &y)
{
    const auto r = __builtin_amdgcn_permlane32_swap(x, y, false, false);
    x = r[0];
    y = r[1];
}
__device__ __forceinline__ void swap_rows(unsigned &x, unsigned &y)
{
    const auto r = __builtin_amdgcn_permlane16_swap(x, y, false, false);
    x = r[0];
    y = r[1];
}
// Row q, block c of v (PER values each) <-> row c, block q, over the four
// 16-lane rows: a lane that held every PER-block of one line holds one block of
// four lines, and back
template <int PER>
__device__ __forceinline__ void transpose_rows(double2 (&v)[4 * PER])
{
    constexpr int ND = 4;  // dwords of a value
#pragma unroll
    for (int p = 0; p < PER; ++p) {
        unsigned a[4][ND];
#pragma unroll
        for (int c = 0; c < 4; ++c) __builtin_memcpy(a[c], &v[c * PER + p], sizeof(double2));
#pragma unroll
        for (int d = 0; d < ND; ++d) {
            swap_halves(a[0][d], a[2][d]);
            swap_halves(a[1][d], a[3][d]);
            swap_rows(a[0][d], a[1][d]);
            swap_rows(a[2][d], a[3][d]);
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) __builtin_memcpy(&v[c * PER + p], a[c], sizeof(double2));
    }
}

// R-point DFT in registers
template <bool INV, int R, class C>
__device__ __forceinline__ void dft_r(C *v)
{
    if constexpr (R == 16) dft16<INV>(v);
    else if constexpr (R == 8) dft8<INV>(v);
    else dft4<INV>(v[0], v[1], v[2], v[3]);
}

// LDS layout of one wavefront's buffer (one mode): base table [base][NZDP],
// z lines [line][LS], transform intermediate [line][LP], transformed products
// [line][TLD], all from slot 0 (each stage's inputs are dead once it stores);
// at the end the wavefront's EMF / stress sums [NACC][NZ] (FP64).  ROWS: the
// z lines stay in registers (rows_inverse, rows_forward)
template <int NZ, class P, class C, bool ROWS_ = false>
struct WaveLayout {
    static constexpr bool ROWS = ROWS_;
    static constexpr int NZD = Dealias<NZ>::nz;
    static constexpr int NZDP = bank_stride(NZD);
    static constexpr int TLD = ROWS ? NZDP : NZD;
    static constexpr int LS = bank_stride(NZ);
    static constexpr int LP = PadIO<NZ, C>::LP;
    static constexpr int cmax(int x, int y) { return x > y ? x : y; }
    static constexpr int RED = (P::NACC * NZ * (int)sizeof(double) + (int)sizeof(C) - 1) / (int)sizeof(C);
    static constexpr int LINES = ROWS ? cmax(P::NLINE, P::NOUT) * LP : P::NLINE * cmax(LS, LP);
    static constexpr int BUF = cmax(cmax(cmax(P::NB * NZDP, LINES), P::NOUT * TLD), RED);
};

// ---------------------------------------------------------------------------
// FP64 transforms at NZ = 128 and 256 whose z lines never leave the registers.
// With NZ = 16 R, k = s + R t and z = j + 16 r,
//   x[z] = sum_s w_R^{-rs} w_NZ^{-js} sum_t w_16^{-jt} X[k]      (inverse)
// and its mirror image forward: a radix-16 pass over t with items (line, s)
// and a radix-R pass over s or r with items (line, j).  In the radix-R pass
// lane (q, j), q its 16-lane row, holds line 4 it + q at z = j + 16 r for
// every r; a transposition over the four rows, in registers, gives it every
// line at the R / 4 points z = j + 16 (q R / 4 + k), where the products are
// formed, and the same transposition leads back.  So a mode takes four passes
// through LDS instead of six (128 instead of 184 b128 accesses per lane at NZ =
// 128) and four exchanges in which the wavefront waits.  Bound by LDS and FP64
// issue at two wavefronts per SIMD.  Measured (HIP events, us, passes through
// LDS before -> now, with what the launch rule's comment says of prefetching):
// MHD_FullQlin 64x128x128 25.9 -> 24.4, 128x128x256 120.8 -> 105.8; MHD_BQlin 25.2 ->
// 23.7, 109.7 -> 101.9; HD_fullU 64x128x128 18.0 -> 16.7.
// ---------------------------------------------------------------------------
template <int NZ, class P>
struct RowPlan {
    static constexpr int R = NZ / 16, PER = R / 4;  // radix, z points per lane
    static constexpr int IX = (P::NLINE + 3) / 4, IO = (P::NOUT + 3) / 4;
    static constexpr int IM = IX > IO ? IX : IO;
    static constexpr int LP = PadIO<NZ, double2>::LP;  // lines of R rows of 17 slots
    static_assert(LP == R * 17, "rows of the intermediate");
    // z point k of a lane
    __device__ static int z(int lane, int k) { return lane % 16 + 16 * (lane / 16 * PER + k); }
    // the radix-16 item of a lane (the last one where it has none), and whether it has one
    template <int NL>
    __device__ static int item(int lane, int it)
    {
        return NL * R % WAVE ? min(lane + it * WAVE, NL * R - 1) : lane + it * WAVE;
    }
    template <int NL>
    __device__ static bool has(int lane, int it)
    {
        return NL * R % WAVE == 0 || lane + it * WAVE < NL * R;
    }
};

// compact spectra in buf ([line][NZDP]) -> the lane's z points of every line,
// X[line / 4][(line % 4) PER + k]; tw(s) = w_NZ^{js}
template <int NZ, class P, class Tw>
__device__ __forceinline__ void rows_inverse(int lane, double2 *buf, const Tw &tw,
                                             double2 (&X)[RowPlan<NZ, P>::IM][NZ / 16])
{
    using D = Dealias<NZ>;
    using RP = RowPlan<NZ, P>;
    constexpr int R = RP::R, LP = RP::LP, NZDP = bank_stride(D::nz), nzl = D::nzl;
    constexpr int IT = (P::NLINE * R + WAVE - 1) / WAVE;
    const int j = lane % 16, q = lane / 16;
    {
        double2 v[IT][16];
#pragma unroll
        for (int it = 0; it < IT; ++it) {
            const int item = RP::template item<P::NLINE>(lane, it), s = item % R;
            const double2 *src = buf + item / R * NZDP;
#pragma unroll
            for (int t = 0; t < 16; ++t) {
                // whether every s of this t is kept, or none, is known here
                const int g = s + R * t;
                if (R * t > nzl && R * t + R - 1 < NZ - nzl) v[it][t] = make_double2(0.0, 0.0);
                else if (R * t + R - 1 <= nzl) v[it][t] = src[g];
                else if (R * t >= NZ - nzl) v[it][t] = src[g - (NZ - D::nz)];
                else v[it][t] = D::kept(g) ? src[D::slot(g)] : make_double2(0.0, 0.0);
            }
        }
        wave_sync();
#pragma unroll
        for (int it = 0; it < IT; ++it) {
            if (it > 0) __builtin_amdgcn_sched_barrier(0);  // one butterfly at a time (registers)
            dft16<true>(v[it]);
            const int item = lane + it * WAVE;
            if (RP::template has<P::NLINE>(lane, it)) {
                double2 *dst = buf + item / R * LP + item % R * 17;
#pragma unroll
                for (int jj = 0; jj < 16; ++jj) dst[jj] = v[it][jj];
            }
        }
    }
    wave_sync();
#pragma unroll
    for (int it = 0; it < RP::IX; ++it) {
        const double2 *src = buf + min(4 * it + q, P::NLINE - 1) * LP + j;
#pragma unroll
        for (int s = 0; s < R; ++s) X[it][s] = src[s * 17];
    }
    wave_sync();
#pragma unroll
    for (int it = 0; it < RP::IX; ++it) {
        if (it > 0) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 1; s < R; ++s) {
            const double2 w = tw(s);
            X[it][s] = cmul(X[it][s], make_double2(w.x, -w.y));
        }
        dft_r<true, R>(X[it]);
        transpose_rows<RP::PER>(X[it]);
    }
}

// the lane's z points of the product lines -> their dealiased spectra in buf,
// [line][NZDP]
template <int NZ, class P, class Tw>
__device__ __forceinline__ void rows_forward(int lane, double2 *buf, const Tw &tw,
                                             double2 (&X)[RowPlan<NZ, P>::IM][NZ / 16])
{
    using D = Dealias<NZ>;
    using RP = RowPlan<NZ, P>;
    constexpr int R = RP::R, LP = RP::LP, NZDP = bank_stride(D::nz), nzl = D::nzl;
    constexpr int IT = (P::NOUT * R + WAVE - 1) / WAVE;
    const int j = lane % 16, q = lane / 16;
#pragma unroll
    for (int it = 0; it < RP::IO; ++it) {
        __builtin_amdgcn_sched_barrier(0);
        transpose_rows<RP::PER>(X[it]);
        dft_r<false, R>(X[it]);
#pragma unroll
        for (int s = 1; s < R; ++s) X[it][s] = cmul(X[it][s], tw(s));
        const int l = 4 * it + q;
        if (P::NOUT % 4 == 0 || l < P::NOUT) {
            double2 *dst = buf + l * LP + j;
#pragma unroll
            for (int s = 0; s < R; ++s) dst[s * 17] = X[it][s];
        }
    }
    wave_sync();
    double2 v[IT][16];
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        const int item = RP::template item<P::NOUT>(lane, it);
        const double2 *src = buf + item / R * LP + item % R * 17;
#pragma unroll
        for (int jj = 0; jj < 16; ++jj) v[it][jj] = src[jj];
    }
    wave_sync();
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        if (it > 0) __builtin_amdgcn_sched_barrier(0);
        dft16<false>(v[it]);
        const int item = lane + it * WAVE, s = item % R;
        if (RP::template has<P::NOUT>(lane, it)) {
            double2 *dst = buf + item / R * NZDP;
#pragma unroll
            for (int t = 0; t < 16; ++t) {
                const int g = s + R * t;
                if (R * t > nzl && R * t + R - 1 < NZ - nzl) continue;
                if (R * t + R - 1 <= nzl) dst[g] = v[it][t];
                else if (R * t >= NZ - nzl) dst[g - (NZ - D::nz)] = v[it][t];
                else if (D::kept(g)) dst[D::slot(g)] = v[it][t];
            }
        }
    }
    wave_sync();
}

template <int NZ, class P, class C>
struct WaveLineSrc {
    const C *sbase;  // [base][NZDP]
    const RealOf<C> *skz;
    __device__ C operator()(int line, int g) const
    {
        using D = Dealias<NZ>;
        if (!D::kept(g)) return Cx<C>::make(0, 0);
        const int m = D::slot(g);
        const C v = sbase[P::base_of(line) * bank_stride(Dealias<NZ>::nz) + m];
        return P::dz_of(line) ? imul(skz[m], v) : v;
    }
};

template <int NZ, class C>
struct WaveCompactDst {
    C *ct;  // [line][nz]
    __device__ void operator()(int line, int j, C v) const
    {
        using D = Dealias<NZ>;
        if (D::kept(j)) ct[line * D::nz + D::slot(j)] = v;
    }
};

// MIXW (C = float2): mixed precision in one launch, each mode in FP64 when
// its flag is set and in FP32 otherwise (no companion launch)
// ALT: the second variant of MHD_BQlin (wave_alt, beside its launch)
template <int NZ, class P, class C, int MODE, int NW, bool SPL, bool MIXW = false, bool ALT = false>
__device__ __forceinline__ void mode_wave_body(const ModeArgs &a)
{
    typedef RealOf<C> R;
    using D = Dealias<NZ>;
    // transforms with the z lines in registers: FP64 at NZ >= 128, HD_fullU's three
    // lines at 128 only (at 256, two wavefronts per SIMD, they need more registers
    // than there are: 47.7 against 46.9 us); not the mixed kernel's FP64 modes, which
    // share their sums by z point with its FP32 ones
    constexpr bool ROWS = sizeof(C) == 16 && !MIXW && !ALT && (NZ == 128 || (NZ > 128 && P::NPAIR == 2));
    using L = WaveLayout<NZ, P, C, ROWS>;
    using PL = Plan2<NZ>;
    constexpr int NZD = D::nz;
    constexpr int KI = (NZD + WAVE - 1) / WAVE;  // kz slots per lane
    constexpr int ZI = (NZ + WAVE - 1) / WAVE;   // z points per lane
    static_assert(KI <= 4 && ZI <= 4, "slots per lane");
    __shared__ C tw[NZ];
    __shared__ R skzr[ROWS ? 1 : NZD];
    __shared__ double skz[NZD];  // FP64 wavenumbers of B and F
    __shared__ R smfz[NZ * P::NMFZ];
    // MIXW: the buffer holds an FP64 mode, and FP64 copies of the tables
    constexpr int BUFC = MIXW ? ((int)(WaveLayout<NZ, P, double2>::BUF * sizeof(double2)) + (int)sizeof(C) - 1) / (int)sizeof(C)
                              : L::BUF;
    __shared__ C wbuf[NW][BUFC > L::BUF ? BUFC : L::BUF];
    __shared__ double2 tw64[MIXW ? NZ : 1];
    __shared__ double smfz64[MIXW ? NZ * P::NMFZ : 1];
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid % WAVE;
    C *buf = wbuf[wave];

    const WgInfo wgi = a.wg[blockIdx.x];
    const int run = wgi.run, g0 = wgi.g0, g1 = wgi.g1, mode_off = wgi.mode_off;
    // AHEAD: a mode's loads, F's of the previous RHS included, at the end of the
    // mode before it, the first ahead of the tables, and the state held for F.  At
    // one slot per lane, where few modes per wavefront leave latency the bound and
    // the registers are there (100 CN steps of 36x60x64 MHD_BQlin with noise 5.93 ->
    // 5.75 ms, the gradient of 200 steps of 32x32x64 30.05 -> 29.48); with more
    // slots they are not (200 steps of 64x128x128 21.8 -> 27.9 ms)
    constexpr bool AHEAD = KI == 1 && (!SPL || MIXW) && !ALT;
    double kxl = 0.0, kyl = 0.0;
    double2 ua[4], na[4];
    auto load_ahead = [&](int l) {
        const int i = mode_off + l;
        kxl = a.kx0[i];
        kyl = a.ky[i];
        const size_t o = (size_t)i * 4 * NZD + min(lane, NZD - 1);
#pragma unroll
        for (int f = 0; f < 2 * P::NPAIR; ++f) {
            ua[f] = a.u[o + f * NZD];
            na[f] = a.n_prev ? a.n_prev[o + f * NZD] : make_double2(0.0, 0.0);
        }
    };
    if constexpr (AHEAD)
        if (g0 + wave < g1) load_ahead(g0 + wave);
    const RunParams rp = a.runs[run];
    const Phys ph = rp.ph;
    const SubTimes st = sub_times<MODE == MODE_CN>(a, run);
    const double linC = to_sgpr(st.linC), nlc1 = to_sgpr(st.nlc1), nlc2 = to_sgpr(st.nlc2);
    const double qt = to_sgpr(rn_mul(ph.q, st.ts)), qdtl = to_sgpr(rn_mul(ph.q, st.dtl));
    const double qt_old = to_sgpr(rn_mul(ph.q, st.tso)), qdtl_old = to_sgpr(rn_mul(ph.q, st.dtlo));
    const double remap_qt = to_sgpr(rn_mul(ph.q, st.tnew));
    const bool do_remap = a.do_remap && rp.remap;

    // shared tables, every load before the first LDS store
    {
        const C *twg = reinterpret_cast<const C *>(sizeof(C) == 8 ? a.tw32 : (const void *)a.tw);
        const double *mfz = a.mfz + (size_t)run * 8 * NZ;
        constexpr int NTH = NW * WAVE;
        constexpr int TWN = (NZ + NTH - 1) / NTH, MFN = (NZ * P::NMFZ + NTH - 1) / NTH;
        static_assert(NZD <= NTH, "one wavenumber per thread");
        C twv[TWN];
        double mfv[MFN];
#pragma unroll
        for (int w = 0; w < TWN; ++w) twv[w] = (tid + w * NTH < NZ) ? twg[tid + w * NTH] : Cx<C>::make(0, 0);
        const double kzt = tid < NZD ? a.kzv[tid] : 0.0;
#pragma unroll
        for (int w = 0; w < MFN; ++w) mfv[w] = (tid + w * NTH < NZ * P::NMFZ) ? mfz[tid + w * NTH] : 0.0;
#pragma unroll
        for (int w = 0; w < TWN; ++w)
            if (tid + w * NTH < NZ) tw[tid + w * NTH] = twv[w];
        if (tid < NZD) {
            if constexpr (!ROWS) skzr[tid] = (R)kzt;
            skz[tid] = kzt;
        }
#pragma unroll
        for (int w = 0; w < MFN; ++w)
            if (tid + w * NTH < NZ * P::NMFZ) smfz[tid + w * NTH] = (R)mfv[w];
        if constexpr (MIXW) {
#pragma unroll
            for (int w = 0; w < TWN; ++w)
                if (tid + w * NTH < NZ) tw64[tid + w * NTH] = a.tw[tid + w * NTH];
#pragma unroll
            for (int w = 0; w < MFN; ++w)
                if (tid + w * NTH < NZ * P::NMFZ) smfz64[tid + w * NTH] = mfv[w];
        }
    }
    // ROWS at NZ = 128: the lane's twiddles, the same for every mode and both
    // directions (28 registers; at NZ = 256 they come from the table)
    constexpr int RT = ROWS && NZ == 128 ? NZ / 16 : 1;
    C twr[RT];
#pragma unroll
    for (int s = 1; s < RT; ++s) twr[s] = reinterpret_cast<const C *>(a.tw)[(lane % 16) * s];
    double acc[ZI][P::NACC];
#pragma unroll
    for (int k = 0; k < ZI; ++k)
#pragma unroll
        for (int c = 0; c < P::NACC; ++c) acc[k][c] = 0.0;
    __syncthreads();

    // the workgroup's modes (run-local l in [g0, g1), one per pass), dealt
    // round robin to its wavefronts; with the mixed-precision split
    // (SPLIT_LO) the FP64 companion takes the modes whose amplitude reaches
    // the threshold
    unsigned long long skip = 0ull;  // SPL: which of the chunk's 64 modes the companion takes
    int cbase = g0 + wave;
    for (int l = g0 + wave; l < g1; l += NW) {
        const int i = mode_off + l;
        if constexpr (SPL && !MIXW) {
            if (a.split == SPLIT_LO) {
                // the flags of this wavefront's next 64 modes, one per lane in
                // one round trip, then read from a ballot
                if ((l - g0 - wave) % (64 * NW) == 0) {
                    const int lq = l + lane * NW;
                    skip = __ballot(lq < g1 && a.hi[mode_off + lq]);
                    cbase = l;
                }
                if ((skip >> ((l - cbase) / NW)) & 1ull) continue;
            }
        }
        // one mode in precision CC (the FP64 or the FP32 transforms), its
        // line buffer and tables
        auto pass = [&](auto ctag, auto *bufc, const auto *twc, const auto *skzrc, const auto *smfzc) {
            using CC = decltype(ctag);
            typedef RealOf<CC> RR;
            using LL = WaveLayout<NZ, P, CC, ROWS>;
            // opaque: keeps what depends on the lane (the profile loads) inside the
            // mode loop instead of in registers across it
            int ln = lane;
            if constexpr (ROWS || (NZ >= 256 && !ALT)) asm volatile("" : "+v"(ln));
            const double kx0 = to_sgpr(AHEAD ? kxl : a.kx0[i]), ky = to_sgpr(AHEAD ? kyl : a.ky[i]);
            const double kx = to_sgpr(rn_add(kx0, rn_mul(qt, ky)));  // kx(t), MHD_FullQlin.cpp:727
            const size_t row = (size_t)i * 4 * NZD;

            // B: 1/lap2, 1/lapF and the base spectral fields (MHD_FullQlin.cpp:220-221,
            // 722-738), fac1D folded in
            // (the loads of every slot of the lane together, one latency; ALT at
            // several slots: each slot's before its use)
            constexpr bool SLOTS = ALT && KI > 1;
            double2 ub[KI][4];
    #pragma unroll
            for (int k = 0; k < KI && !SLOTS; ++k) {
                const size_t o = row + min(lane + k * WAVE, NZD - 1);
    #pragma unroll
                for (int f = 0; f < 4; ++f) {
                    if (f >= 2 * P::NPAIR) ub[k][f] = make_double2(0.0, 0.0);
                    else if constexpr (AHEAD) ub[k][f] = ua[f];
                    else ub[k][f] = a.u[o + f * NZD];
                }
            }
    #pragma unroll
            for (int k = 0; k < KI; ++k) {
                if (k > 0) __builtin_amdgcn_sched_barrier(0);  // one slot at a time (registers)
                const int m = lane + k * WAVE;
                if (KI * WAVE == NZD || m < NZD) {
                    if constexpr (SLOTS) {
    #pragma unroll
                        for (int f = 0; f < 4; ++f)
                            ub[k][f] = f < 2 * P::NPAIR ? a.u[row + f * NZD + m] : make_double2(0.0, 0.0);
                    }
                    const double2 u0 = ub[k][0], u1 = ub[k][1], u2 = ub[k][2], u3 = ub[k][3];
                    const double kzk = skz[m], kz2 = -(kzk * kzk);
                    const bool zero = (ky == 0.0 && m == 0);
                    const double lap2 = zero ? 0.0 : (-ky * ky + kz2);
                    const double ilap2 = zero ? 1.0 : 1.0 / lap2;
                    P::bases(u0, u1, u2, u3, kx, ky, kzk, ilap2, a.fac, bufc + m, LL::NZDP);
                }
            }
            wave_sync();

            // F's loads (the state again, the previous substep's RHS) ahead of the
            // forward transforms where registers are left for them: at one wavefront
            // per SIMD (128x128x256: 114.6 -> 104.3 us) and for HD_fullU's half state at
            // NZ = 128 (17.2 -> 16.8); elsewhere they spill (33.6 against 24.3 us at NZ = 128)
            constexpr bool EARLY = P::NPAIR == 1 ? ROWS && NZ == 128 : NZ >= 256 && !ALT;
            double2 uf[EARLY ? KI : 1][4], nf[EARLY ? KI : 1][4];
            auto load_early = [&]() {
    #pragma unroll
                for (int k = 0; k < KI; ++k) {
                    const size_t o = row + min(ln + k * WAVE, NZD - 1);
    #pragma unroll
                    for (int f = 0; f < 2 * P::NPAIR; ++f) {
                        uf[k][f] = a.u[o + f * NZD];
                        nf[k][f] = a.n_prev ? a.n_prev[o + f * NZD] : make_double2(0.0, 0.0);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            };
            // ModelBQ's dz uz constant of a ky = 0 mode: i kx fac1D ux at kz = 0
            auto dz_const = [&]() {
                return from_d<CC>(ky == 0.0 ? imul(kx, cscale(a.fac, a.u[row])) : make_double2(0.0, 0.0));
            };
            // the EMF / stress terms of z point k, and its product lines through put(line, value)
            auto products = [&](int k, int zz, CC dzc, const CC *x, int ld, const auto &put) {
                const double ftfac = (ky == 0.0 ? 1.0 : 2.0) * rp.rsf;  // MHD_FullQlin.cpp:314-318
                RR mfl[P::NMFZ];
    #pragma unroll
                for (int c = 0; c < P::NMFZ; ++c) mfl[c] = smfzc[c * NZ + zz];
                CC prod[2][3];
                double racc[2][2];
                P::products(0, x, ld, mfl, (RR)kx, (RR)ky, dzc, prod[0], racc[0]);
                P::products(1, x, ld, mfl, (RR)kx, (RR)ky, dzc, prod[1], racc[1]);
    #pragma unroll
                for (int part = 0; part < 2; ++part) {
                    acc[k][P::acc_slot(part, 0)] += ftfac * racc[part][0];
                    if (P::NACC == 4) acc[k][P::acc_slot(part, 1)] += ftfac * racc[part][1];
                }
    #pragma unroll
                for (int part = 0; part < 2; ++part)
    #pragma unroll
                    for (int c = 0; c < 3; ++c)
                        if (c < P::nprod(part)) put(P::out_line(part, c), prod[part][c]);
            };
            if constexpr (ROWS) {
                using RP = RowPlan<NZ, P>;
                const auto tws = [&](int s) {
                    if constexpr (RT > 1) return twr[s];
                    else return twc[ln % 16 * s];
                };
                CC X[RP::IM][RP::R];
                rows_inverse<NZ, P>(ln, bufc, tws, X);
                // D: products in registers
                const CC dzc = dz_const();
    #pragma unroll
                for (int k = 0; k < ZI; ++k) {
                    if (k > 0) __builtin_amdgcn_sched_barrier(0);  // one z point at a time (registers)
                    CC x[P::NLINE];
    #pragma unroll
                    for (int l = 0; l < P::NLINE; ++l) x[l] = X[l / 4][l % 4 * RP::PER + k];
                    products(k, RP::z(ln, k), dzc, x, 1, [&](int l, CC v) { X[l / 4][l % 4 * RP::PER + k] = v; });
                }
                if constexpr (EARLY) load_early();
                // E
                rows_forward<NZ, P>(ln, bufc, tws, X);
            } else {
                // C: inverse transforms of the padded lines
                {
                    const PadIO<NZ, CC> pad{bufc};
                    wave_pass<NZ, P::NLINE, true, PL::R1, 1>(lane, twc, WaveLineSrc<NZ, P, CC>{bufc, skzrc}, pad);
                    wave_pass<NZ, P::NLINE, true, PL::R2, PL::R1>(lane, twc, pad, BufIO<LL::LS, CC>{bufc});
                }
                // D: products on the z grid, in place, and the EMF / stress sums
                const CC dzc = dz_const();
    #pragma unroll
                for (int k = 0; k < ZI; ++k) {
                    if (k > 0) __builtin_amdgcn_sched_barrier(0);  // one z point at a time (registers)
                    const int zz = lane + k * WAVE;
                    if (ZI * WAVE == NZ || zz < NZ) {
                        CC *X = bufc + zz;
                        products(k, zz, dzc, X, LL::LS, [&](int l, CC v) { X[l * LL::LS] = v; });
                    }
                }
                wave_sync();
                if constexpr (EARLY) load_early();

                // E: forward transforms of the product lines, dealiased band kept
                {
                    const PadIO<NZ, CC> pad{bufc};
                    wave_pass<NZ, P::NOUT, false, PL::R1, 1>(lane, twc, BufIO<LL::LS, CC>{bufc}, pad);
                    wave_pass<NZ, P::NOUT, false, PL::R2, PL::R1>(lane, twc, pad, WaveCompactDst<NZ, CC>{bufc});
                }
            }

            // F: RHS, dissipation operator at the substep end, update
            bool hit = false;
            if (do_remap) hit = remap_hit(remap_qt, rp.remap_thr, kx0, ky);
    #pragma unroll
            for (int k = 0; k < KI; ++k) {
                // one slot at a time: the scheduler would otherwise hoist the
                // loads of every slot of the lane and run out of registers
                if (k > 0) __builtin_amdgcn_sched_barrier(0);
                const int m = lane + k * WAVE;
                if (!(KI * WAVE == NZD || m < NZD)) continue;
                const size_t off = row + m;
                const double kzk = skz[m], kz2 = -(kzk * kzk);
                // 1/lapF as in B (recomputed rather than held through the transforms)
                const double lap2 = (ky == 0.0 && m == 0) ? 0.0 : (-ky * ky + kz2);
                const double ilapF = (l == 0 && m == 0) ? 1.0 : 1.0 / (-kx * kx + lap2);
                double2 U0, U1, U2 = make_double2(0.0, 0.0), U3 = U2, np[4];
                if constexpr (EARLY) {
                    U0 = uf[k][0];
                    U1 = uf[k][1];
                    if constexpr (P::NPAIR == 2) {
                        U2 = uf[k][2];
                        U3 = uf[k][3];
                    }
    #pragma unroll
                    for (int f = 0; f < 2 * P::NPAIR; ++f) np[f] = nf[k][f];
                } else if constexpr (AHEAD) {
                    U0 = ua[0];
                    U1 = ua[1];
                    if constexpr (P::NPAIR == 2) {
                        U2 = ua[2];
                        U3 = ua[3];
                    }
    #pragma unroll
                    for (int f = 0; f < 2 * P::NPAIR; ++f) np[f] = na[f];
                } else {
                    U0 = a.u[off];
                    U1 = a.u[off + NZD];
                    if constexpr (P::NPAIR == 2) {
                        U2 = a.u[off + 2 * NZD];
                        U3 = a.u[off + 3 * NZD];
                    }
    #pragma unroll
                    for (int f = 0; f < 2 * P::NPAIR; ++f) np[f] = a.n_prev ? a.n_prev[off + f * NZD] : make_double2(0.0, 0.0);
                }
                const CC *T = bufc + m;
                const double kxn = kx + qdtl * ky;
                const double opn = P::op((-kxn * kxn - ky * ky) + kz2, ph);
                double opo = 0.0;
                if constexpr (MODE == MODE_CN) {
                    // the "old" operator is the one of the previous substep (or
                    // linearOPs_Init at t0)
                    const double kxo = rn_add(kx0, rn_mul(qt_old, ky)), kxe = kxo + qdtl_old * ky;
                    opo = P::op(st.oinit ? -kxo * kxo + lap2 : (-kxe * kxe - ky * ky) + kz2, ph);
                }
    #pragma unroll
                for (int pr = 0; pr < P::NPAIR; ++pr) {
                    double2 N0, N1;
                    P::rhs_pair(pr, T, LL::TLD, U0, U1, U2, U3, kx, ky, kzk, ilapF, ph, N0, N1);
                    const double Ln = P::lin(pr, opn, ph);
                    const size_t off0 = off + (2 * pr) * NZD, off1 = off0 + NZD;
                    if constexpr (MODE == MODE_RHS) {
                        if (a.n_out) {
                            a.n_out[off0] = N0;
                            a.n_out[off1] = N1;
                        }
                        if (a.lin_out) a.lin_out[off0] = a.lin_out[off1] = Ln;
                        continue;
                    }
                    const double2 u0 = pr ? U2 : U0, u1 = pr ? U3 : U1;
                    const double2 p0 = np[2 * pr], p1 = np[2 * pr + 1];
                    double2 un0, un1;
                    if constexpr (MODE == MODE_ELIN) {
                        // RK3CN_Elin.cpp:303-305, :335-337, :368-370
                        const double e = exp(linC * Ln);
                        double2 s0 = cscale(nlc1, N0), s1 = cscale(nlc1, N1);
                        if (a.n_prev) {
                            s0 = cadd(s0, cscale(nlc2, p0));
                            s1 = cadd(s1, cscale(nlc2, p1));
                        }
                        un0 = cscale(e, cadd(s0, u0));
                        un1 = cscale(e, cadd(s1, u1));
                    } else {
                        // RK3CN.cpp:105-107, :141-143, :177-179
                        const double Lo = P::lin(pr, opo, ph);
                        const double denom = 1.0 / (1.0 - linC * Ln);
                        const double c1 = nlc1 * denom, co = (1 + linC * Lo) * denom;
                        double2 s0 = cscale(c1, N0), s1 = cscale(c1, N1);
                        if (a.n_prev) {
                            const double c2 = nlc2 * denom;
                            s0 = cadd(s0, cscale(c2, p0));
                            s1 = cadd(s1, cscale(c2, p1));
                        }
                        un0 = cadd(s0, cscale(co, u0));
                        un1 = cadd(s1, cscale(co, u1));
                    }
                    if (hit) un0 = un1 = make_double2(0.0, 0.0);
                    a.u_out[off0] = un0;
                    a.u_out[off1] = un1;
                    if (a.n_out) {
                        a.n_out[off0] = N0;
                        a.n_out[off1] = N1;
                    }
                }
            }
            if (hit && lane == 0) a.kx0[i] = rn_sub(kx0, rp.remap_shift);
        };
        if constexpr (MIXW) {
            // mixed precision per mode: the flagged modes in FP64 in this
            // same launch, the others in FP32, both in the wavefront's buffer
            if (a.split == SPLIT_LO && a.hi[i])
                pass(double2{}, reinterpret_cast<double2 *>(buf), tw64, skz, smfz64);
            else
                pass(C{}, buf, tw, skzr, smfz);
        } else {
            pass(C{}, buf, tw, skzr, smfz);
        }
        if constexpr (AHEAD)
            if (l + NW < g1) load_ahead(l + NW);
        // the next mode's B overwrites the transformed products F read
        wave_sync();
    }

    // fixed-order reduction of the wavefronts' sums: one partial [NACC][NZ]
    // per workgroup
    __syncthreads();
    double *red = reinterpret_cast<double *>(&wbuf[0][0]);
    static_assert(NW * P::NACC * NZ * sizeof(double) <= sizeof(wbuf), "reduction fits the buffers");
#pragma unroll
    for (int k = 0; k < ZI; ++k) {
        int zz = lane + k * WAVE;
        if constexpr (ROWS) zz = RowPlan<NZ, P>::z(lane, k);
        if (ZI * WAVE == NZ || zz < NZ)
#pragma unroll
            for (int c = 0; c < P::NACC; ++c) red[(wave * P::NACC + c) * NZ + zz] = acc[k][c];
    }
    __syncthreads();
    for (int k = tid; k < P::NACC * NZ; k += NW * WAVE) {
        double s = 0.0;
#pragma unroll
        for (int w = 0; w < NW; ++w) s += red[w * P::NACC * NZ + k];
        a.partials[(size_t)blockIdx.x * P::NACC * NZ + k] = s;
    }
}

// MHD_FullQlin (ModelFull), MHD_BQlin (ModelBQ) and HD_fullU (ModelHD); workgroups of
// mode_waves(NZ) wavefronts: 8 at NZ <= 128 (one workgroup per CU at NZ = 128
// in FP64: 116 KB of LDS; measured at 64x128x128 in an earlier build: 8
// wavefronts and 252 workgroups 31.1 us, 4 and 504 31.9 us, 2 and 1008 31.6 us and twice the
// partial rows for the column reduction), 4 at NZ = 256 (26 KB per wavefront
// in FP64, one wavefront per SIMD with the whole register file)
// (the velocity-only policy, with 3 lines per transform, keeps 8 at NZ = 256)
template <class P>
constexpr int mode_waves(int NZ) { return NZ >= 256 && P::NPAIR == 2 ? 4 : 8; }
template <class P>
constexpr int wave_occ(int NZ) { return NZ >= 256 && P::NPAIR == 2 ? 1 : 2; }
template <int NZ, class P, int MODE, bool ALT = false>
__global__ __launch_bounds__(mode_waves<P>(NZ) * WAVE) __attribute__((amdgpu_waves_per_eu(wave_occ<P>(NZ))))
void k_wave64(ModeArgs a)
{
    mode_wave_body<NZ, P, double2, MODE, mode_waves<P>(NZ), false, false, ALT>(a);
}
template <int NZ, class P, int MODE, bool ALT = false>
__global__ __launch_bounds__(mode_waves<P>(NZ) * WAVE) __attribute__((amdgpu_waves_per_eu(wave_occ<P>(NZ))))
void k_wave32(ModeArgs a)
{
    mode_wave_body<NZ, P, float2, MODE, mode_waves<P>(NZ), true, false, ALT>(a);
}
template <int NZ, class P, int MODE, bool ALT = false>
__global__ __launch_bounds__(mode_waves<P>(NZ) * WAVE) __attribute__((amdgpu_waves_per_eu(wave_occ<P>(NZ))))
void k_wave_mix(ModeArgs a)
{
    mode_wave_body<NZ, P, float2, MODE, mode_waves<P>(NZ), true, true, ALT>(a);
}

}  // namespace qlk
