// Per-size-class part of the batched implicit integrator.  The host emits
// this text once per system size class, inside a namespace, after defining
// _numeq_, SODECL_LPO (lanes per orbit, a power of two; 64 / SODECL_LPO orbits
// share a wavefront) and SODECL_BR (rows per lane) for that class and including the system plugin
// there.
//
// One orbit is integrated by SODECL_LPO lanes of a wavefront.  Two forms:
//   * windowed (SODECL_WINDOW): the plugin evaluates component i from its
//     neighbours up to SODE_REACH away (sode_system_window,
//     calc_jacobian_band_window).  A lane owns SODECL_BR consecutive
//     components, and the state, residual, band and solve stay in its
//     registers; only the SODE_REACH outermost components at either end move
//     to the neighbouring lanes (DPP wavefront shifts).  No LDS, and what the
//     plugin gives as constant zeros in the band drops out at compile time.
//   * through LDS, for any component function: components are owned strided
//     (comp = lane + LPO c) for the right-hand side, the band Jacobian and the
//     Newton update, and the solve reads its rows back from LDS.
// In both, the tridiagonal solve of each Newton iteration runs in parallel over
// contiguous row partitions (lane k owns rows [kR, kR + R)): elimination
// inside each partition expresses its rows through the last unknown of the
// previous partition and its own last unknown, the resulting tridiagonal
// system in those LPO unknowns is solved by parallel cyclic reduction across
// lanes, and the partition rows follow by substitution.
// The matrix is the one the reference's tridiagonal sweep solves
// (ie.cl:10-48, im.cl:3-41): sub-diagonal a_i = J[i][i+1] for i < N-2 (0
// otherwise), diagonal J[i][i], super-diagonal c_i = J[i+1][i] (c_{N-1} = 0),
// each entry already scaled to I + s*dt*J.  Solving it by partitions instead
// of one sweep changes only the rounding.

#define SODECL_OPW (SODECL_BG / SODECL_LPO)                   // orbits per wavefront
// Every lane owns exactly SODECL_BR components / rows: the bounds tests below are then compile-time true.
#define SODECL_FULL (_numeq_ == SODECL_LPO * SODECL_BR)
#define SODECL_OWNS(comp) (SODECL_FULL || (comp) < _numeq_)
// Row c of this lane's partition exists.
#define SODECL_ROW(c) (SODECL_FULL || r0 + (c) < _numeq_)
// LDS index of row i in the solve's arrays.  A 64-bit LDS access serves 16
// lanes per pass over 32 four-byte banks, so 16 doubles that differ modulo
// 16 are conflict-free.  The lanes of the solve read row j of their own
// partitions (rows kR + j, a stride of R), the strided owners write and
// read consecutive rows: rotating each block of 16 rows by its block index
// keeps both patterns conflict-free (measured: bank-conflict cycles from
// 0.12 to 0.01 of LDS cycles) without padding, so the rows stay N long.
#if SODECL_BR >= 2
#define SODECL_TI(i) (((i) & ~15) | (((i) + ((i) >> 4)) & 15))
#define SODECL_TLEN ((_numeq_ + 15) / 16 * 16)
#else
#define SODECL_TI(i) (i)
#define SODECL_TLEN (_numeq_)
#endif
// LDS doubles per orbit (the form through LDS): four rows -- the evaluation point, which the
// right-hand side of the solve (then its solution) overwrites once the
// Jacobian has read it, and the three band rows -- and the parameters when
// there are more than 8 (fewer stay in registers).  16 KiB for 512
// equations, so that ten wavefronts fit a CU's LDS.
#define SODECL_PLDS (_numpar_ <= 8 ? 0 : _numpar_)
#define SODECL_ORBIT_LDS (4 * SODECL_TLEN + SODECL_PLDS)

// The values of lanes l - 32 (up) and l + 32 (down), 0 past either end of
// the wavefront, from one half-wavefront swap (v_permlane32_swap) per 32-bit
// half: with both operands v, its first result holds lane l mod 32's value
// and its second lane 32 + l mod 32's.
SODECL_INLINE void sodecl_pcr_pair32(double v, int lane, double& up, double& down)
{
    const long long b = __double_as_longlong(v);
    const auto lo = __builtin_amdgcn_permlane32_swap((int)(b & 0xffffffffll), (int)(b & 0xffffffffll), false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap((int)(b >> 32), (int)(b >> 32), false, false);
    const double from_low = __longlong_as_double(((long long)(int)hi[0] << 32) | (long long)(unsigned int)lo[0]);
    const double from_high = __longlong_as_double(((long long)(int)hi[1] << 32) | (long long)(unsigned int)lo[1]);
    up = lane >= 32 ? from_low : 0.0;
    down = lane < 32 ? from_high : 0.0;
}

// v of orbit lane - s (up) or lane + s (down), 0 past either end of the
// orbit's lanes.  Orbits of 16 lanes are DPP rows: row shifts, which bring
// 0 past either end by themselves (smaller orbits drop what crossed over
// from the neighbouring one).  Otherwise distances of one and two are DPP
// wavefront shifts (with a whole wavefront per orbit the shift brings 0 past
// either end; 32-lane orbits drop what crossed over), longer ones a bpermute.
SODECL_INLINE double sodecl_pcr_neighbour(double v, int lane, int s, bool up)
{
    const bool inside = up ? lane - s >= 0 : lane + s < SODECL_LPO;
#if SODECL_LPO <= 16
    double w;
    switch (s) {
    case 1: w = up ? sodecl_dpp<SODECL_DPP_ROW_SHR(1)>(v) : sodecl_dpp<SODECL_DPP_ROW_SHL(1)>(v); break;
    case 2: w = up ? sodecl_dpp<SODECL_DPP_ROW_SHR(2)>(v) : sodecl_dpp<SODECL_DPP_ROW_SHL(2)>(v); break;
    case 4: w = up ? sodecl_dpp<SODECL_DPP_ROW_SHR(4)>(v) : sodecl_dpp<SODECL_DPP_ROW_SHL(4)>(v); break;
    default: w = up ? sodecl_dpp<SODECL_DPP_ROW_SHR(8)>(v) : sodecl_dpp<SODECL_DPP_ROW_SHL(8)>(v); break;
    }
    return (SODECL_LPO == 16 || inside) ? w : 0.0;
#else
    if (s <= 2) {
        double w = up ? sodecl_dpp<SODECL_DPP_WAVE_SHR1>(v) : sodecl_dpp<SODECL_DPP_WAVE_SHL1>(v);
        if (s == 2) w = up ? sodecl_dpp<SODECL_DPP_WAVE_SHR1>(w) : sodecl_dpp<SODECL_DPP_WAVE_SHL1>(w);
        return (SODECL_LPO == 64 || inside) ? w : 0.0;
    }
    const double w = up ? __shfl_up(v, (unsigned)s, SODECL_LPO) : __shfl_down(v, (unsigned)s, SODECL_LPO);
    return inside ? w : 0.0;
#endif
}

// v of the wavefront's previous (up) or next lane: row shifts where orbits lie
// within 16-lane rows, else wavefront shifts.
SODECL_INLINE double sodecl_shift(double v, bool up)
{
#if SODECL_LPO <= 16
    return up ? sodecl_dpp<SODECL_DPP_ROW_SHR(1)>(v) : sodecl_dpp<SODECL_DPP_ROW_SHL(1)>(v);
#else
    return up ? sodecl_dpp<SODECL_DPP_WAVE_SHR1>(v) : sodecl_dpp<SODECL_DPP_WAVE_SHL1>(v);
#endif
}

// Sum over the orbit's lanes, the same value on each of them.
SODECL_INLINE double sodecl_orbit_sum(double v)
{
    double s[1] = {v};
    sodecl_lane_sums<SODECL_LPO>(s);
    return s[0];
}

// Partitions that hold rows, and the cyclic-reduction levels they need
// (ceil(log2(partitions)); inactive partitions are identity rows).
#define SODECL_NPART ((_numeq_ + SODECL_BR - 1) / SODECL_BR)
#define SODECL_PCR_LEVELS (SODECL_NPART > 32 ? 6 : SODECL_NPART > 16 ? 5 : SODECL_NPART > 8 ? 4 : \
                           SODECL_NPART > 4 ? 3 : SODECL_NPART > 2 ? 2 : SODECL_NPART > 1 ? 1 : 0)

// Solves M x = v for the matrix above.  Row j of this lane's partition has the
// sub-diagonal up(j), diagonal di(j) and super-diagonal lo(j) (functions, so that
// rows in LDS are read where they are used), with the reference's zeros in place
// (a_i = 0 outside 1 <= i < N-2, c_{N-1} = 0); rows past the last are identity
// rows (0, 1, 0) with v = 0, so that every partition is complete.  All lanes of
// the wavefront, lane = the lane's index within its orbit.
template <class Lo, class Di, class Up, class V>
SODECL_INLINE void sodecl_tri_solve(Lo lo, Di di, Up up, V v, double (&x)[SODECL_BR], int lane)
{
    const int R = SODECL_BR, I = R > 1 ? R - 1 : 1;   // R - 1 interior rows, then the partition's last
    double ia[I], be[I], ga[I];   // ia = 1/alpha
    double e[I], f[I], g[I];
    // forward elimination through the interior, tracking the coupling to
    // x_L = last unknown of the previous partition
#pragma unroll
    for (int j = 0; j < R - 1; ++j) {
        double al = di(j);
        if (j == 0) {
            be[0] = v(0);
            ga[0] = up(0);
        } else if (sodecl_zero(up(j))) {
            be[j] = v(j);
            ga[j] = 0.0;
        } else {
            const double m = up(j) * ia[j - 1];
            if (!sodecl_zero(lo(j - 1))) al = di(j) - m * lo(j - 1);
            be[j] = v(j) - m * be[j - 1];
            ga[j] = sodecl_zero(ga[j - 1]) ? 0.0 : -m * ga[j - 1];
        }
        ia[j] = sodecl_rcp(al);
    }
    // backward: interior x_i = e_i + f_i x_L + g_i x_R, x_R = own last unknown
#pragma unroll
    for (int j = R - 2; j >= 0; --j) {
        const double ci = lo(j);
        f[j] = sodecl_zero(ga[j]) ? 0.0 : -ga[j] * ia[j];
        if (j == R - 2) {
            e[j] = be[j] * ia[j];
            g[j] = sodecl_zero(ci) ? 0.0 : -ci * ia[j];
        } else if (sodecl_zero(ci)) {
            e[j] = be[j] * ia[j];
            g[j] = 0.0;
        } else {
            e[j] = (be[j] - ci * e[j + 1]) * ia[j];
            if (!sodecl_zero(f[j + 1])) f[j] = (-ga[j] - ci * f[j + 1]) * ia[j];
            g[j] = sodecl_zero(g[j + 1]) ? 0.0 : (-ci * g[j + 1]) * ia[j];
        }
    }
    // reduced row of partition k (its last row): A X_{k-1} + B X_k + C X_{k+1} = D.
    // Without interior the row before the last is X_{k-1} itself, and a
    // partition's first row is its X.
    const double e_last = R > 1 ? e[I - 1] : 0.0, f_last = R > 1 ? f[I - 1] : 1.0, g_last = R > 1 ? g[I - 1] : 0.0;
    double A = 0.0, B = di(R - 1), C = 0.0, D = v(R - 1);
    if (!sodecl_zero(up(R - 1))) {
        A = up(R - 1) * f_last;
        B = B + up(R - 1) * g_last;
        D = D - up(R - 1) * e_last;
    }
    if (!sodecl_zero(lo(R - 1))) {
        // the next partition's first row, through X_k and X_{k+1}
        B = B + lo(R - 1) * sodecl_pcr_neighbour(R > 1 ? f[0] : 0.0, lane, 1, false);
        C = lo(R - 1) * sodecl_pcr_neighbour(R > 1 ? g[0] : 1.0, lane, 1, false);
        D = D - lo(R - 1) * sodecl_pcr_neighbour(R > 1 ? e[0] : 0.0, lane, 1, false);
    }
    // When every reduced row is already decoupled (A = C = 0: the partition
    // boundaries fall where the matrix has no coupling, as for a system of
    // 2x2 blocks such as the Brusselator chain under the reference's index
    // mapping), cyclic reduction would leave B and D unchanged: skip it.
    if (!(sodecl_zero(A) && sodecl_zero(C)) && !__all(A == 0.0 && C == 0.0)) {
        // parallel cyclic reduction over the reduced rows.  Each lane shares its
        // row scaled by its pivot's reciprocal (A/B, C/B, D/B), so one
        // reciprocal per lane and level and three values per direction suffice:
        // with the neighbours m = lane - s and p = lane + s,
        //   A' = -A (A/B)_m,  C' = -C (C/B)_p,
        //   B' = B - A (C/B)_m - C (A/B)_p,  D' = D - A (D/B)_m - C (D/B)_p;
        // rows past either end contribute nothing (shared values 0).
#pragma unroll
        for (int lv = 0; lv < SODECL_PCR_LEVELS; ++lv) {
            const int s = 1 << lv;
            const double iB = sodecl_rcp(B);
            const double a = A * iB, c = C * iB, d = D * iB;
            double am, cm, dm, ap, cp, dp;
            if (SODECL_LPO == 64 && s == 32) {
                sodecl_pcr_pair32(a, lane, am, ap);
                sodecl_pcr_pair32(c, lane, cm, cp);
                sodecl_pcr_pair32(d, lane, dm, dp);
            } else {
                am = sodecl_pcr_neighbour(a, lane, s, true);
                cm = sodecl_pcr_neighbour(c, lane, s, true);
                dm = sodecl_pcr_neighbour(d, lane, s, true);
                ap = sodecl_pcr_neighbour(a, lane, s, false);
                cp = sodecl_pcr_neighbour(c, lane, s, false);
                dp = sodecl_pcr_neighbour(d, lane, s, false);
            }
            const double nB = B - A * cm - C * ap;
            const double nD = D - A * dm - C * dp;
            A = -A * am;
            C = -C * cp;
            B = nB;
            D = nD;
        }
    }
    const double X = D * sodecl_rcp(B);
    const double Xm = sodecl_pcr_neighbour(X, lane, 1, true);
#pragma unroll
    for (int j = 0; j < R - 1; ++j) {
        x[j] = e[j];
        if (!sodecl_zero(f[j])) x[j] = x[j] + f[j] * Xm;
        if (!sodecl_zero(g[j])) x[j] = x[j] + g[j] * X;
    }
    x[R - 1] = X;
}

#if SODECL_WINDOW
// Two-level matrices: every row that is coupled to another is coupled only to
// rows without couplings (known from the constant zeros; row 0 stands for the
// next partition's and row R - 1 for the previous one's).  A chain of cells
// with two species each has this form under the reference's index mapping.
// Nothing needs eliminating then: every pivot is its diagonal element, the
// uncoupled rows divide, and the others substitute.
template <class Lo, class Up> SODECL_INLINE bool sodecl_two_level(Lo lo, Up up)
{
    const int R = SODECL_BR;
    const auto leaf = [&](int j) { return sodecl_zero(up(j)) && sodecl_zero(lo(j)); };
    bool two = true;
#pragma unroll
    for (int j = 0; j < R; ++j)
        two = two && ((sodecl_zero(up(j)) || leaf((j + R - 1) % R)) && (sodecl_zero(lo(j)) || leaf((j + 1) % R)));
    return two;
}
SODECL_INLINE bool sodecl_normal(double v) { return __builtin_amdgcn_class(v, 0x108); }
// Changes a and b to such that their reciprocals were b/q and a/q, where a b is
// no normal number: each one's power of two goes to the other; a zero, an
// infinity or no number gets no number, as from its own reciprocal.
SODECL_INLINE void sodecl_pivots_scaled(double* pa, double* pb, double* q)
{
    const double a = *pa, b = *pb;
    const bool na = __builtin_amdgcn_class(a, 0x267), nb = __builtin_amdgcn_class(b, 0x267);   // zero, infinite, NaN
    const double fa = na ? 1.0 : __builtin_amdgcn_frexp_mant(a), fb = nb ? 1.0 : __builtin_amdgcn_frexp_mant(b);
    *q = fa * fb;
    *pb = na ? __builtin_nan("") : __builtin_amdgcn_ldexp(fb, -__builtin_amdgcn_frexp_exp(a));
    *pa = nb ? __builtin_nan("") : __builtin_amdgcn_ldexp(fa, -__builtin_amdgcn_frexp_exp(b));
}
// Solves such a system: every row as if it were uncoupled, then the coupled ones
// from their neighbours' (uncoupled) values.  Which rows are coupled only saves
// work here: a zero that is not seen as a constant at one of the tests costs a
// product with it.  The reciprocals come in pairs, 1/a = b/(ab) and
// 1/b = a/(ab): ten issue slots in place of fourteen (a reciprocal's estimate
// takes four).  An orbit whose residual norm is no number gets no numbers (the
// reference's sweep carries it through every row).  Against the general solve:
// 236 instead of 256 issue slots per Newton iteration of eight rows, 32768
// Brusselator chains of 32, 128 and 512 equations 8.50 -> 7.68 ms.
template <class Lo, class Up>
SODECL_INLINE void sodecl_two_level_solve(Lo lo, double (&di)[SODECL_BR], Up up, double (&v)[SODECL_BR], double err,
                                          double (&x)[SODECL_BR], int lane)
{
    const int R = SODECL_BR, P = R > 1 ? R / 2 : 1;
    double q[P];   // 1/di[j] = di[j ^ 1] / q[j / 2]
    bool plain = !(err != err);
    if (R == 1) q[0] = di[0];
#pragma unroll
    for (int k = 0; k < R / 2; ++k) {
        q[k] = di[2 * k] * di[2 * k + 1];
        plain = plain & sodecl_normal(q[k]);
    }
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(!plain) != 0, 0)) {
#pragma unroll
        for (int j = 0; j < R; ++j) v[j] = err != err ? err : v[j];
#pragma unroll
        for (int k = 0; k < R / 2; ++k)
            if (!sodecl_normal(q[k])) sodecl_pivots_scaled(&di[2 * k], &di[2 * k + 1], &q[k]);
    }
#pragma unroll
    for (int k = 0; k < P; ++k) q[k] = sodecl_rcp(q[k]);
    const auto inv = [&](int j) { return R > 1 ? di[(j ^ 1) % R] * q[j / 2] : q[0]; };
    double u[R];
#pragma unroll
    for (int j = 0; j < R; ++j) u[j] = v[j] * inv(j);
    double before = 0.0, after = 0.0;   // the neighbouring partitions' last and first unknown
    if (!sodecl_zero(up(0))) before = sodecl_pcr_neighbour(u[R - 1], lane, 1, true);
    if (!sodecl_zero(lo(R - 1))) after = sodecl_pcr_neighbour(u[0], lane, 1, false);
#pragma unroll
    for (int j = 0; j < R; ++j) {
        x[j] = u[j];
        if (!(sodecl_zero(up(j)) && sodecl_zero(lo(j)))) {
            double s = v[j];
            if (!sodecl_zero(up(j))) s = s - up(j) * (j > 0 ? u[j - 1 < 0 ? 0 : j - 1] : before);
            if (!sodecl_zero(lo(j))) s = s - lo(j) * (j + 1 < R ? u[j + 1 < R ? j + 1 : 0] : after);
            x[j] = s * inv(j);
        }
    }
}
#endif

// The most steps of any orbit of the wavefront, in a scalar register.
SODECL_INLINE int sodecl_wave_steps(int steps)
{
#pragma unroll
    for (int m = SODECL_LPO; m < 64; m <<= 1) steps = max(steps, __shfl_xor(steps, m));
    return __builtin_amdgcn_readfirstlane(steps);
}

// The routine is inlined into its class's kernel (a called function gets
// only half of the register budget from hipRTC as VGPRs and moves values
// through AGPRs: 50 AGPR reads per Newton iteration of the 512-equation
// class, 10% more VALU instructions).
#ifndef SODECL_BATCH_ITEM_ATTR
#define SODECL_BATCH_ITEM_ATTR __attribute__((always_inline))
#endif
// Integrates the orbits of one work item -- SODECL_OPW orbits, item[k] on the k-th group of SODECL_LPO lanes (item[k] < 0: none) -- for steps[o]
// steps of implicit Euler (SODECL_SOLVER 3, ie.cl:50-117) or implicit
// midpoint (4, im.cl:43-118) with the reference's Newton iteration: stop
// when the L1 (IE) / L2 (IM) residual norm is below _epsilon1_, at most
// SODECL_NEWTON_MAXIT updates.  Snapshot j (state after j * _numsteps_
// steps) goes to out[ooff[o] + j * neq ...]; newton[o] receives the updates
// taken.  The orbits of a wavefront run in lockstep: the wavefront steps
// until its longest orbit is done and iterates until every orbit's Newton
// iteration has stopped; an orbit that has stopped computes along on its
// last values without storing them or counting updates.
#if SODECL_WINDOW
__device__ SODECL_BATCH_ITEM_ATTR void sodecl_batch_item(const int* __restrict__ item, const int* __restrict__ steps_of,
                                  const long long* __restrict__ yoff, const long long* __restrict__ ooff,
                                  const double* __restrict__ y0_all, const double* __restrict__ params_all,
                                  double* __restrict__ out_all, long long* __restrict__ newton, double* lds)
{
    static_assert(SODECL_BR >= SODE_REACH, "a component's neighbours sit on the next lane at most");
    const int part = threadIdx.x / SODECL_LPO;
    const int lane = threadIdx.x % SODECL_LPO;
    const int r0 = lane * SODECL_BR;
    const int o = item[part];
    const bool has = o >= 0;
    const int steps = has ? steps_of[o] : 0;
    const int smax = sodecl_wave_steps(steps);
    // parameters in registers when there are few, else in LDS
#if _numpar_ <= 8
    (void)lds;
    double sh_p[_numpar_ > 0 ? _numpar_ : 1];
#pragma unroll
    for (int k = 0; k < _numpar_; ++k) sh_p[k] = has ? params_all[(size_t)o * _numpar_ + k] : 0.0;
#else
    // (an odd row length: orbits of a wavefront read different banks)
    double* const sh_p = lds + (size_t)part * (_numpar_ | 1);
    for (int k = lane; k < _numpar_; k += SODECL_LPO) sh_p[k] = has ? params_all[(size_t)o * _numpar_ + k] : 0.0;
    sodecl_wave_sync();
#endif
    double* const out = has ? out_all + ooff[o] : nullptr;
    double y[SODECL_BR], gg[SODECL_BR];
#pragma unroll
    for (int c = 0; c < SODECL_BR; ++c) {
        y[c] = 0.0;
        if (has && SODECL_ROW(c)) {
            y[c] = y0_all[yoff[o] + r0 + c];
            out[r0 + c] = y[c];
        }
    }
    double t = 0.0;
    long long updates = 0;
#if SODECL_SOLVER == 3
    const double scale = -1.00;
#else
    const double scale = -0.50;
#endif
    for (int s = 0; s < smax; ++s) {
        const bool live = s < steps;
#pragma unroll
        for (int c = 0; c < SODECL_BR; ++c) gg[c] = y[c];
        for (int it = 0; it < SODECL_NEWTON_MAXIT; ++it) {
            // the evaluation point of this lane's components and SODE_REACH
            // more on either side
            double win[SODECL_BR + 2 * SODE_REACH];
#pragma unroll
            for (int c = 0; c < SODECL_BR; ++c) {
#if SODECL_SOLVER == 3
                win[SODE_REACH + c] = gg[c];
#else
                win[SODE_REACH + c] = (y[c] + gg[c]) * 0.5;
#endif
            }
#pragma unroll
            for (int d = 0; d < SODE_REACH; ++d) {
                // (what crosses over from another orbit stands for components
                // that do not exist)
                win[d] = sodecl_shift(win[SODECL_BR + d], true);
                win[SODE_REACH + SODECL_BR + d] = sodecl_shift(win[SODE_REACH + d], false);
            }
            double r[SODECL_BR], lo[SODECL_BR], di[SODECL_BR], up[SODECL_BR], x[SODECL_BR];
            double err = 0.0;
#pragma unroll
            for (int c = 0; c < SODECL_BR; ++c) {
                r[c] = 0.0;
                if (SODECL_ROW(c)) {
                    const double fv = sode_system_window(r0 + c, t, &win[SODE_REACH + c], sh_p);
                    r[c] = gg[c] - y[c] - fv * _m_dt_;
#if SODECL_SOLVER == 3
                    err = err + fabs(r[c]);
#else
                    err = err + r[c] * r[c];
#endif
                }
            }
            // The band does not depend on the residual norm: evaluated while
            // the reduction and vote are in flight; not used in the iteration
            // that ends a step.
#pragma unroll
            for (int c = 0; c < SODECL_BR; ++c) {
                lo[c] = 0.0;
                di[c] = 1.0;
                up[c] = 0.0;
                if (SODECL_ROW(c)) {
                    double l, d, u;
                    calc_jacobian_band_window(r0 + c, &win[SODE_REACH + c], sh_p, &l, &d, &u);
                    // a_i = J[i][i+1] for 1 <= i < N-2, c_i = J[i+1][i] for i < N-1, else 0
                    if (!sodecl_zero(l)) lo[c] = r0 + c < _numeq_ - 1 ? l * scale * _m_dt_ : 0.0;
                    if (!sodecl_zero(u)) up[c] = (r0 + c >= 1 && r0 + c < _numeq_ - 2) ? u * scale * _m_dt_ : 0.0;
                    di[c] = d * scale * _m_dt_ + 1;
                }
            }
            err = sodecl_orbit_sum(err);
#if SODECL_SOLVER == 3
            const bool done = !live || err < _epsilon1_;
#else
            // sqrt(err) < _epsilon1_ without the root, which the whole wavefront
            // waited for (450 chains of 5 to 100 cells, Newton run to
            // convergence: 468 -> 419 us)
            const bool done = !live || err < SODECL_EPSILON1_SQUARED;
#endif
            if (__all(done)) break;
            const auto low = [&](int j) { return lo[j]; };
            const auto upp = [&](int j) { return up[j]; };
            if (sodecl_two_level(low, upp)) {
                sodecl_two_level_solve(low, di, upp, r, err, x, lane);
            } else {
                // A residual that is not a number leaves no component a number
                // (the reference's sweep carries it through every row).
                if (__builtin_expect(__builtin_amdgcn_ballot_w64(err != err) != 0, 0)) {
#pragma unroll
                    for (int c = 0; c < SODECL_BR; ++c) r[c] = err != err ? err : r[c];
                }
                sodecl_tri_solve(low, [&](int j) { return di[j]; }, upp, [&](int j) { return r[j]; }, x, lane);
            }
            if (!done) {
#pragma unroll
                for (int c = 0; c < SODECL_BR; ++c) gg[c] = gg[c] - x[c];
                ++updates;
            }
        }
        if (live) {
#pragma unroll
            for (int c = 0; c < SODECL_BR; ++c) y[c] = gg[c];
        }
        t = t + _m_dt_;
        if (live && (s + 1) % _numsteps_ == 0) {
            double* o_snap = out + (size_t)((s + 1) / _numsteps_) * _numeq_;
#pragma unroll
            for (int c = 0; c < SODECL_BR; ++c)
                if (SODECL_ROW(c)) o_snap[r0 + c] = y[c];
        }
    }
    if (has && lane == 0) newton[o] = updates;
}
#else
__device__ SODECL_BATCH_ITEM_ATTR void sodecl_batch_item(const int* __restrict__ item, const int* __restrict__ steps_of,
                                  const long long* __restrict__ yoff, const long long* __restrict__ ooff,
                                  const double* __restrict__ y0_all, const double* __restrict__ params_all,
                                  double* __restrict__ out_all, long long* __restrict__ newton, double* lds)
{
    const int part = threadIdx.x / SODECL_LPO;
    const int lane = threadIdx.x % SODECL_LPO;
    const int o = item[part];
    const bool has = o >= 0;
    const int steps = has ? steps_of[o] : 0;
    const int smax = sodecl_wave_steps(steps);
    double* const sh_g = lds + (size_t)part * SODECL_ORBIT_LDS;   // evaluation point (g, or (y+g)/2), plain layout
    double* const sh_r = sh_g;   // then the residual -> right-hand side -> solution (rotated layout)
    double* const sh_lo = sh_r + SODECL_TLEN;
    double* const sh_di = sh_lo + SODECL_TLEN;
    double* const sh_up = sh_di + SODECL_TLEN;
#if _numpar_ <= 8
    // few parameters: a register copy, which the plugin's reads need not
    // reload from LDS after every store of the band rows
    double sh_p[_numpar_ > 0 ? _numpar_ : 1];
#pragma unroll
    for (int k = 0; k < _numpar_; ++k) sh_p[k] = has ? params_all[(size_t)o * _numpar_ + k] : 0.0;
#else
    double* const sh_p = sh_up + SODECL_TLEN;
    for (int k = lane; k < _numpar_; k += SODECL_LPO) sh_p[k] = has ? params_all[(size_t)o * _numpar_ + k] : 0.0;
#endif
    double* const out = has ? out_all + ooff[o] : nullptr;
    double y[SODECL_BR], gg[SODECL_BR];
#pragma unroll
    for (int c = 0; c < SODECL_BR; ++c) {
        const int comp = lane + c * SODECL_LPO;
        y[c] = 0.0;
        if (has && SODECL_OWNS(comp)) {
            y[c] = y0_all[yoff[o] + comp];
            out[comp] = y[c];
        }
    }
    double t = 0.0;
    long long updates = 0;
#if SODECL_SOLVER == 3
    const double scale = -1.00;
#else
    const double scale = -0.50;
#endif
    for (int s = 0; s < smax; ++s) {
        const bool live = s < steps;
#pragma unroll
        for (int c = 0; c < SODECL_BR; ++c) gg[c] = y[c];
        for (int it = 0; it < SODECL_NEWTON_MAXIT; ++it) {
            // The orbit's lanes sit in this wavefront (SODECL_BG is one
            // wavefront): wavefront-scope ordering of the LDS accesses suffices.
            sodecl_wave_sync();   // previous readers of sh_g are done
#pragma unroll
            for (int c = 0; c < SODECL_BR; ++c) {
                const int comp = lane + c * SODECL_LPO;
#if SODECL_SOLVER == 3
                if (SODECL_OWNS(comp)) sh_g[comp] = gg[c];
#else
                if (SODECL_OWNS(comp)) sh_g[comp] = (y[c] + gg[c]) * 0.5;
#endif
            }
            sodecl_wave_sync();
            double r[SODECL_BR];
            double err = 0.0;
#pragma unroll
            for (int c = 0; c < SODECL_BR; ++c) {
                const int comp = lane + c * SODECL_LPO;
                r[c] = 0.0;
                if (SODECL_OWNS(comp)) {
                    const double fv = sode_system_i(comp, t, sh_g, sh_p);
                    r[c] = gg[c] - y[c] - fv * _m_dt_;
#if SODECL_SOLVER == 3
                    err = err + fabs(r[c]);
#else
                    err = err + r[c] * r[c];
#endif
                }
            }
            // The band Jacobian and the right-hand side go to LDS before the
            // residual norm is known: they do not depend on it, and computing
            // them while the wavefront-wide reduction and vote are in flight
            // hides those (IE 254 -> 228 ms, IM 229 -> 223 ms on the
            // benchmark batch); in the iteration that ends a step they are
            // not used.
#pragma unroll
            for (int c = 0; c < SODECL_BR; ++c) {
                const int comp = lane + c * SODECL_LPO;
                if (SODECL_OWNS(comp)) {
                    double lo, di, up;
                    calc_jacobian_band_i(comp, sh_g, sh_p, &lo, &di, &up);
                    // a_i = J[i][i+1] for 1 <= i < N-2, c_i = J[i+1][i] for i < N-1, else 0
                    sh_lo[SODECL_TI(comp)] = comp < _numeq_ - 1 ? lo * scale * _m_dt_ : 0.0;
                    sh_up[SODECL_TI(comp)] = (comp >= 1 && comp < _numeq_ - 2) ? up * scale * _m_dt_ : 0.0;
                    sh_di[SODECL_TI(comp)] = di * scale * _m_dt_ + 1;
                }
            }
            sodecl_wave_sync();   // every read of the evaluation point is done
#pragma unroll
            for (int c = 0; c < SODECL_BR; ++c) {
                const int comp = lane + c * SODECL_LPO;
                if (SODECL_OWNS(comp)) sh_r[SODECL_TI(comp)] = r[c];
            }
            err = sodecl_orbit_sum(err);
#if SODECL_SOLVER == 3
            const bool done = !live || err < _epsilon1_;
#else
            const bool done = !live || err < SODECL_EPSILON1_SQUARED;
#endif
            if (__all(done)) break;
            sodecl_wave_sync();
            {
                // this lane's partition, the solution written back in place
                double px[SODECL_BR];
                const int r0 = lane * SODECL_BR;
                auto row = [&](const double* a, int j, double past) {
                    return SODECL_FULL || r0 + j < _numeq_ ? a[SODECL_TI(r0 + j)] : past;
                };
                sodecl_tri_solve([&](int j) { return row(sh_lo, j, 0.0); }, [&](int j) { return row(sh_di, j, 1.0); },
                                 [&](int j) { return row(sh_up, j, 0.0); }, [&](int j) { return row(sh_r, j, 0.0); }, px,
                                 lane);
#pragma unroll
                for (int j = 0; j < SODECL_BR; ++j)
                    if (SODECL_FULL || r0 + j < _numeq_) sh_r[SODECL_TI(r0 + j)] = px[j];
            }
            sodecl_wave_sync();
            if (!done) {
#pragma unroll
                for (int c = 0; c < SODECL_BR; ++c) {
                    const int comp = lane + c * SODECL_LPO;
                    if (SODECL_OWNS(comp)) gg[c] = gg[c] - sh_r[SODECL_TI(comp)];
                }
                ++updates;
            }
        }
        if (live) {
#pragma unroll
            for (int c = 0; c < SODECL_BR; ++c) y[c] = gg[c];
        }
        t = t + _m_dt_;
        if (live && (s + 1) % _numsteps_ == 0) {
            double* o_snap = out + (size_t)((s + 1) / _numsteps_) * _numeq_;
#pragma unroll
            for (int c = 0; c < SODECL_BR; ++c) {
                const int comp = lane + c * SODECL_LPO;
                if (SODECL_OWNS(comp)) o_snap[comp] = y[c];
            }
        }
    }
    if (has && lane == 0) newton[o] = updates;
}
#endif  // SODECL_WINDOW

#undef SODECL_OPW
#undef SODECL_PLDS
#undef SODECL_ORBIT_LDS
#undef SODECL_TI
#undef SODECL_TLEN
#undef SODECL_NPART
#undef SODECL_PCR_LEVELS
#undef SODECL_FULL
#undef SODECL_OWNS
#undef SODECL_ROW
