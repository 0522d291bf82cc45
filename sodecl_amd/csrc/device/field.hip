// Field form of the group schedule: drifts that couple an orbit's components
// through a few sums over all of them,
//   f_i = F(i, t, y_i, p, phi(y_i), S),   S_k = sum_j phi_k(y_j),  k < SODE_FIELDS
// (the all-to-all sine coupling is one: sum_j sin(y_j - y_i) =
// S_sin cos y_i - S_cos sin y_i).  A plugin that defines
//   void sode_field(int i, double t, double yi, double ps[], double po[], double phi[SODE_FIELDS])
//   double sode_system_field(int i, double t, double yi, double ps[], double po[], double phi[], double sum[])
//   int sode_field_own_param(int i, int k)
// is integrated with O(N) work per drift instead of the O(N^2) of the
// per-component and pairwise forms.  ps are the first SODE_FIELD_SHARED
// parameters, po the SODE_FIELD_OWN parameters of component i,
// po[k] = p[sode_field_own_param(i, k)].  The integration passes nothing through LDS:
// SODECL_FL lanes share an orbit, lane l owns the SODECL_FC consecutive
// components from l * SODECL_FC on, states and parameters in registers, sums
// its features over them and then over the lanes by DPP moves, which leave
// the same bits on every lane.
//
// What bounds it: the VALU issue of the features' evaluation (for the sine
// coupling one sine and cosine per component and drift).  Several components
// per lane make the reduction (three instructions per field and level) a small
// part and give each wavefront independent chains; a launch too small to fill
// the chip so takes one component per lane (sodecl_capi.cpp chooses).
//
// Euler-Maruyama runs here when each component's diffusion reads only its own
// state and its own noise (double sode_system_stoch_own(int i, double t,
// double yi, double ps[], double po[], double zi), as many noises as components): a lane
// draws the Threefry calls of its own components.  With one component per lane
// the two lanes of a call's pair draw two steps' noise and swap halves.
#if SODECL_SCHEDULE == 2 && SODECL_USE_FIELD

#define SODECL_FOPB (SODECL_FBLOCK / SODECL_FL)
// lanes that own components, and the power of two of lanes their sums span
#define SODECL_FROWS ((_numeq_ + SODECL_FC - 1) / SODECL_FC)
#define SODECL_FWIDTH (SODECL_FROWS > 32 ? 64 : SODECL_FROWS > 16 ? 32 : SODECL_FROWS > 8 ? 16 : \
                       SODECL_FROWS > 4 ? 8 : SODECL_FROWS > 2 ? 4 : SODECL_FROWS > 1 ? 2 : 1)
#define SODECL_FSTAGES (SODECL_SOLVER == 2 ? 4 : 1)
// lengths of the parameter arrays (never 0)
#define SODECL_FPS (SODE_FIELD_SHARED > 0 ? SODE_FIELD_SHARED : 1)
#define SODECL_FPO (SODE_FIELD_OWN > 0 ? SODE_FIELD_OWN : 1)
static_assert(SODECL_FROWS <= SODECL_FL, "every component has a lane");
static_assert(!SODECL_IS_SDE || (SODECL_FC == 1 ? SODECL_FL > 1 : SODECL_FC % 2 == 0),
              "a noise pair belongs to one lane, or to two of the orbit's");

// Component c of this lane exists (compile-time true when the lanes' shares
// come out even and no lane is spare).
#define SODECL_FOWNS(c)                                                                          \
    (SODECL_FROWS * SODECL_FC == _numeq_ ? (SODECL_FROWS == SODECL_FL || lane < SODECL_FROWS)    \
                                         : lane * SODECL_FC + (c) < _numeq_)
// Its index, 0 where it does not exist (results discarded).
#define SODECL_FINDEX(c) (SODECL_FOWNS(c) ? lane * SODECL_FC + (c) : 0)

// The parameters of one orbit that this lane's components read.
struct sodecl_field_params {
    double ps[SODECL_FPS];
    double po[SODECL_FC][SODECL_FPO];
};
SODECL_INLINE void sodecl_field_load_params(const double* p, bool active, int lane, sodecl_field_params& q)
{
#pragma unroll
    for (int k = 0; k < SODE_FIELD_SHARED; ++k) q.ps[k] = active && k < _numpar_ ? p[k] : 0.0;
#pragma unroll
    for (int c = 0; c < SODECL_FC; ++c)
#pragma unroll
        for (int k = 0; k < SODE_FIELD_OWN; ++k) {
            const unsigned m = (unsigned)sode_field_own_param(SODECL_FINDEX(c), k);
            q.po[c][k] = active && SODECL_FOWNS(c) && m < _numpar_ ? p[m] : 0.0;
        }
}

// Which orbit of the block a thread works on, and its lane there.  From 32
// lanes on the sums over lanes start with two products of the matrix cores with
// ones (v_mfma_f64_4x4x4_4b_f64 holds four 4 x 4 matrices, matrix b on the
// lanes with l / 4 mod 4 = b): the first adds the four lanes of a column, the
// second the four columns, and lane moves join the orbit's two or four
// matrices.  1500 orbits of 33 components on 32 lanes, 300 RK4 steps: 373 ->
// 354 us; on 16 lanes the two products take as long as the four levels of moves
// and lane moves stay.
#define SODECL_FMATRIX (SODECL_FL >= 32)
SODECL_INLINE int sodecl_field_lane(int tid)
{
    if (SODECL_FL == 32) return (tid & 7) | ((tid >> 1) & 24);
    return tid % SODECL_FL;
}
SODECL_INLINE int sodecl_field_slot(int tid)
{
    if (SODECL_FL == 32) return (tid >> 6) * 2 + ((tid >> 3) & 1);
    return tid / SODECL_FL;
}

// Sums over the orbit's lanes (lanes without components hold zeros), the same
// bits on each, the fields side by side (each level waits for the one before).
template <int K>
SODECL_INLINE void sodecl_field_reduce(double (&v)[K])
{
#if SODECL_FMATRIX
#pragma unroll
    for (int k = 0; k < K; ++k) v[k] = __builtin_amdgcn_mfma_f64_4x4x4f64(v[k], 1.0, 0.0, 0, 0, 0);
#pragma unroll
    for (int k = 0; k < K; ++k) v[k] = __builtin_amdgcn_mfma_f64_4x4x4f64(1.0, v[k], 0.0, 0, 0, 0);
#pragma unroll
    for (int k = 0; k < K; ++k)   // matrices 0 and 1 (2 and 3): lanes i and 7 - i
        v[k] = v[k] + sodecl_dpp<SODECL_DPP_HALF_MIRROR>(v[k]);
    if (SODECL_FL == 64) {
#pragma unroll
        for (int k = 0; k < K; ++k) v[k] = v[k] + sodecl_dpp<SODECL_DPP_MIRROR>(v[k]);
    }
#else
    sodecl_lane_sums<SODECL_FWIDTH>(v);
#endif
}

// The features' sums over the orbit's components.
SODECL_INLINE void sodecl_field_sums(int lane, const double (&phi)[SODECL_FC][SODE_FIELDS], double (&sum)[SODE_FIELDS])
{
#pragma unroll
    for (int k = 0; k < SODE_FIELDS; ++k) {
        sum[k] = SODECL_FOWNS(0) ? phi[0][k] : 0.0;
#pragma unroll
        for (int c = 1; c < SODECL_FC; ++c) sum[k] = sum[k] + (SODECL_FOWNS(c) ? phi[c][k] : 0.0);
    }
    sodecl_field_reduce(sum);
}

// Features, their sums, and the drift of this lane's components at x.
// A source that defines SODE_FIELD_MARKED_SINCOS promises that a NaN sine from
// any sincos() of its sode_field makes a sum NaN (no comparison, selection,
// minimum or maximum takes it in between).  Its features come from a copy of
// the source whose sincos() gives a NaN sine where the library's function is
// needed (sodecl_sincos_marked): no branch or library code per component, one
// test of the sums per drift.  Sums that are not numbers send the orbit's features
// through the source as it stands, one component at a time.
SODECL_INLINE void sodecl_field_eval(double t, const double (&x)[SODECL_FC], sodecl_field_params& pp, int lane,
                                     double (&phi)[SODECL_FC][SODE_FIELDS], double (&sum)[SODE_FIELDS],
                                     double (&f)[SODECL_FC])
{
#ifdef SODECL_FIELD_MARKED
#pragma unroll
    for (int c = 0; c < SODECL_FC; ++c) sodecl_marked::sode_field(SODECL_FINDEX(c), t, x[c], pp.ps, pp.po[c], phi[c]);
    sodecl_field_sums(lane, phi, sum);
    bool bad = false;
#pragma unroll
    for (int k = 0; k < SODE_FIELDS; ++k) bad = bad || sum[k] != sum[k];
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(bad) != 0, 0)) {
#pragma unroll 1
        for (int q = 0; q < SODECL_FC; ++q) {
            double xq = x[0], po[SODECL_FPO], one[SODE_FIELDS];
#pragma unroll
            for (int k = 0; k < SODE_FIELD_OWN; ++k) po[k] = pp.po[0][k];
#pragma unroll
            for (int c = 1; c < SODECL_FC; ++c) {
                xq = c == q ? x[c] : xq;
#pragma unroll
                for (int k = 0; k < SODE_FIELD_OWN; ++k) po[k] = c == q ? pp.po[c][k] : po[k];
            }
            sode_field(SODECL_FINDEX(q), t, xq, pp.ps, po, one);
#pragma unroll
            for (int c = 0; c < SODECL_FC; ++c)
#pragma unroll
                for (int k = 0; k < SODE_FIELDS; ++k) phi[c][k] = c == q ? one[k] : phi[c][k];
        }
        sodecl_field_sums(lane, phi, sum);
    }
#else
#pragma unroll
    for (int c = 0; c < SODECL_FC; ++c) sode_field(SODECL_FINDEX(c), t, x[c], pp.ps, pp.po[c], phi[c]);
    sodecl_field_sums(lane, phi, sum);
#endif
#pragma unroll
    for (int c = 0; c < SODECL_FC; ++c) f[c] = sode_system_field(SODECL_FINDEX(c), t, x[c], pp.ps, pp.po[c], phi[c], sum);
}

#if SODECL_SOLVER == 1
// Euler (euler.cl:10-18)
SODECL_INLINE void sodecl_field_step(double t, double (&y)[SODECL_FC], sodecl_field_params& pp, int lane)
{
    double phi[SODECL_FC][SODE_FIELDS], sum[SODE_FIELDS], f[SODECL_FC];
    sodecl_field_eval(t, y, pp, lane, phi, sum, f);
#pragma unroll
    for (int c = 0; c < SODECL_FC; ++c) y[c] = y[c] + f[c] * _m_dt_;
}
#elif SODECL_SOLVER == 2
// Classic RK4 (rk4.cl:17-64)
SODECL_INLINE void sodecl_field_step(double t, double (&y)[SODECL_FC], sodecl_field_params& pp, int lane)
{
    double phi[SODECL_FC][SODE_FIELDS], sum[SODE_FIELDS], f[SODECL_FC], acc[SODECL_FC], x[SODECL_FC];
    sodecl_field_eval(t, y, pp, lane, phi, sum, f);
#pragma unroll
    for (int c = 0; c < SODECL_FC; ++c) {
        acc[c] = f[c];
        x[c] = y[c] + (_m_dt_ * 0.50) * f[c];
    }
    sodecl_field_eval(t + 0.50 * _m_dt_, x, pp, lane, phi, sum, f);
#pragma unroll
    for (int c = 0; c < SODECL_FC; ++c) {
        acc[c] = acc[c] + 2.00 * f[c];
        x[c] = y[c] + (_m_dt_ * 0.50) * f[c];
    }
    sodecl_field_eval(t + 0.50 * _m_dt_, x, pp, lane, phi, sum, f);
#pragma unroll
    for (int c = 0; c < SODECL_FC; ++c) {
        acc[c] = acc[c] + 2.00 * f[c];
        x[c] = y[c] + _m_dt_ * f[c];
    }
    sodecl_field_eval(t + _m_dt_, x, pp, lane, phi, sum, f);
#pragma unroll
    for (int c = 0; c < SODECL_FC; ++c) y[c] = y[c] + SODECL_RK4_UPDATE(acc[c] + f[c]);
}
#else
// Euler-Maruyama (stochastic_euler.cl:10-22) with this lane's noise z.
SODECL_INLINE void sodecl_field_step(double t, double (&y)[SODECL_FC], sodecl_field_params& pp, int lane,
                                     const double (&z)[SODECL_FC])
{
    double phi[SODECL_FC][SODE_FIELDS], sum[SODE_FIELDS], f[SODECL_FC];
    sodecl_field_eval(t, y, pp, lane, phi, sum, f);
#pragma unroll
    for (int c = 0; c < SODECL_FC; ++c) {
        const double gn = sode_system_stoch_own(SODECL_FINDEX(c), t, y[c], pp.ps, pp.po[c], z[c]);
        y[c] = y[c] + f[c] * _m_dt_ + gn;
    }
}
#endif

// Workspace rows of the adjoint: the state before each step, [orbit][step][neq],
// then t of each step, [orbit][step], both behind the same pointer (the sweep
// evaluates the stages again, whose features its vector-Jacobian products
// need anyway, so a row is a quarter of RK4's four stage vectors).
SODECL_INLINE void sodecl_field_store(double* ws, size_t rows, size_t row, double t, const double (&y)[SODECL_FC],
                                      int lane)
{
#pragma unroll
    for (int c = 0; c < SODECL_FC; ++c)
        if (SODECL_FOWNS(c)) ws[row * _numeq_ + lane * SODECL_FC + c] = y[c];
    ws[rows * _numeq_ + row] = t;   // the same value from every lane, which each reads back itself
}

// Integration kernel: arguments and outputs as sodecl_group's.
extern "C" __global__ void __launch_bounds__(SODECL_FBLOCK) SODECL_KERNEL_ATTR
sodecl_field(double* __restrict__ t_state, double* __restrict__ y_state, const double* __restrict__ params,
             double* __restrict__ counters, double* __restrict__ traj, long long* __restrict__ newton,
             int orbits, int s0, int nseg, int final_snap, double* __restrict__ ckpt_t,
             double* __restrict__ ckpt_y, int ckpt_every, long long gstep0, double* __restrict__ stage_ws,
             long long ws_steps)
{
    SODECL_EXP_TABLE_INIT();
    const int lane = sodecl_field_lane(threadIdx.x);
    const int slot = sodecl_field_slot(threadIdx.x);
    const int orbit = blockIdx.x * SODECL_FOPB + slot;
    const bool active = orbit < orbits;
    (void)newton;
    sodecl_field_params pp;
    sodecl_field_load_params(params + (size_t)orbit * _numpar_, active, lane, pp);
    double y[SODECL_FC];
#pragma unroll
    for (int c = 0; c < SODECL_FC; ++c)
        y[c] = (active && SODECL_FOWNS(c)) ? y_state[(size_t)orbit * _numeq_ + lane * SODECL_FC + c] : 1.0;
    double t = active ? t_state[orbit] : 0.0;
    const size_t slab = (size_t)_numeq_ * (size_t)orbits;
    long long g = gstep0;
    // checkpoint k is the state before global step k * ckpt_every
    long long ck = ckpt_y ? (gstep0 + ckpt_every - 1) / ckpt_every : 0;
    long long ck_step = ck * ckpt_every;
#if SODECL_IS_SDE
    double cnt = active ? counters[orbit] : 0.0;
    const double dtsqrt = sqrt(_m_dt_);
    // Counters that stay whole numbers below 2^53 advance as 64-bit integers
    // (the doubles' sums are exact there); any other counter takes the
    // reference's addition of each call.
    const long long all_calls = (long long)nseg * _numsteps_ * SODECL_CALLS;
    const bool whole = sodecl_counters_whole(cnt, (double)all_calls);
    const double after = sodecl_counter_after(cnt, all_calls, whole);
    // this lane's next call: its pair's, of the next step from odd lanes with
    // one component per lane
    cnt = sodecl_counter_after(cnt, SODECL_FC == 1 ? (lane >> 1) + ((lane & 1) ? SODECL_CALLS : 0) : lane * SODECL_FC / 2, whole);
    sodecl_u64 word = sodecl_counter_word(cnt);
    (void)stage_ws;
    (void)ws_steps;
#if SODECL_FC == 1
    bool drawn = false;     // this step's noise was drawn with the previous step's
    double znext = 0.0;
#endif
#endif

    for (int s = 0; s < nseg; ++s) {
        if (traj && active) {
#pragma unroll
            for (int c = 0; c < SODECL_FC; ++c)
                if (SODECL_FOWNS(c))
                    traj[(size_t)(s0 + s) * slab + (size_t)(lane * SODECL_FC + c) * orbits + orbit] = y[c];
        }
        // the segment's steps in runs that end at the next checkpoint, so that
        // the step loop tests only its count
        for (int it = 0; it < _numsteps_;) {
            int run = _numsteps_ - it;
            if (ckpt_y) {
                if (g == ck_step) {
                    const long long k = ck++;
                    ck_step += ckpt_every;
                    if (active) {
#pragma unroll
                        for (int c = 0; c < SODECL_FC; ++c)
                            if (SODECL_FOWNS(c))
                                ckpt_y[(size_t)k * slab + (size_t)(lane * SODECL_FC + c) * orbits + orbit] = y[c];
                        if (lane == 0) ckpt_t[(size_t)k * orbits + orbit] = t;
                    }
                }
                if (ck_step - g < run) run = (int)(ck_step - g);   // g < ck_step here
            }
            const int end = it + run;
#if SODECL_IS_SDE
            // (two copies of the step: the branch in one cost 1.3%)
            const auto step = [&](const bool ints) __attribute__((always_inline)) {
                double z[SODECL_FC];
#if SODECL_FC == 1
                // Lane l draws call l / 2 of this step (l even) or of the next
                // one (l odd): each lane of a call's pair keeps its half of the
                // step it drew and swaps the other.
                if (!drawn) {
                    double z0, z1;
                    sodecl_noise_pair(orbit, word, dtsqrt, &z0, &z1);
                    word += 2 * SODECL_CALLS;
                    if (!ints) {
                        cnt = sodecl_counter_after(cnt, 2 * SODECL_CALLS, false);
                        word = sodecl_counter_word(cnt);
                    }
                    // (lanes l and l ^ 1 are neighbours in every mapping)
                    const double other = sodecl_dpp<SODECL_DPP_XOR1>((lane & 1) ? z0 : z1);
                    z[0] = (lane & 1) ? other : z0;
                    znext = (lane & 1) ? z1 : other;
                } else {
                    z[0] = znext;
                }
                drawn = !drawn;
#else
                sodecl_u64 w[SODECL_FC / 2];
#pragma unroll
                for (int c = 0; c < SODECL_FC / 2; ++c) w[c] = word + (sodecl_u64)c;
                word += SODECL_CALLS;
                if (!ints) {
#pragma unroll
                    for (int c = 0; c < SODECL_FC / 2; ++c) {
                        w[c] = sodecl_counter_word(cnt);
                        cnt = cnt + 1;
                    }
                    cnt = sodecl_counter_after(cnt, SODECL_CALLS - SODECL_FC / 2, false);
                }
#pragma unroll
                for (int c = 0; c < SODECL_FC; c += 2) sodecl_noise_pair(orbit, w[c / 2], dtsqrt, &z[c], &z[c + 1]);
#endif
                sodecl_field_step(t, y, pp, lane, z);
                t = t + _m_dt_;
            };
            if (whole)
                for (; it < end; ++it, ++g) step(true);
            else
                for (; it < end; ++it, ++g) step(false);
#else
            if (stage_ws) {
                const size_t rows = (size_t)orbits * (size_t)ws_steps;
                for (; it < end; ++it, ++g) {
                    if (active) sodecl_field_store(stage_ws, rows, (size_t)orbit * ws_steps + g, t, y, lane);
                    sodecl_field_step(t, y, pp, lane);
                    t = t + _m_dt_;
                }
            } else {
                it = end;
                g += run;
                const auto step = [&]() {
                    sodecl_field_step(t, y, pp, lane);
                    t = t + _m_dt_;
                };
#if SODECL_FC == 1 && SODECL_SOLVER == 1
                // one component per lane is what launches of few wavefronts take,
                // where the loop's scalar instructions count: four steps in a block
                // (1024 orbits of 10 components x 420 steps 96 -> 92 us with two,
                // 88 with four)
                for (; run > 3; run -= 4) {
                    step();
                    step();
                    step();
                    step();
                }
#endif
                for (; run > 0; --run) step();
            }
#endif
        }
    }
    if (active) {
#pragma unroll
        for (int c = 0; c < SODECL_FC; ++c) {
            if (SODECL_FOWNS(c)) {
                const int comp = lane * SODECL_FC + c;
                if (traj && final_snap) traj[(size_t)(s0 + nseg) * slab + (size_t)comp * orbits + orbit] = y[c];
                y_state[(size_t)orbit * _numeq_ + comp] = y[c];
            }
        }
        if (lane == 0) {
            t_state[orbit] = t;
#if SODECL_IS_SDE
            counters[orbit] = after;
#endif
        }
    }
}

// ---------------------------------------------------------------------------
// Discrete adjoint in field form (Euler, RK4): the transpose of the steps
// above, checkpointed or from a whole-run workspace like
// sodecl_group_adjoint.  Of a step only its first state is kept: the sweep
// evaluates the step's stages once more (the features and sums each product
// needs) and then walks them backwards in registers.  With lam the
// cotangent of f,
//   Sbar_k = sum_i lam_i dF_i/dS_k                             (group sums)
//   lam^T df/dy_i = lam_i dF_i/dy_i + sum_k (lam_i dF_i/dphi_k + Sbar_k) dphi_k/dy_i
// from the plugin's
//   void sode_field_vjp_sum(i, t, yi, ps, po, phi[], sum[], lam, sbar[])     adds to sbar[k]
//   double sode_field_vjp(i, t, yi, ps, po, phi[], sum[], sbar[], lam)
//   void sode_field_vjp_params(i, t, yi, ps, po, phi[], sum[], lam, gs[], go[])
// the last adding lam df_i/dp for the shared and the component's own parameters
// to gs and go; other parameters have no gradient.
// ---------------------------------------------------------------------------
#if defined(SODECL_ADJOINT) && (SODECL_SOLVER == 1 || SODECL_SOLVER == 2)

// gx = (df/dy)^T l at the point whose features and sums are given; parameter
// products are added to grad.
SODECL_INLINE void sodecl_field_product(double t, const double (&x)[SODECL_FC], const double (&phi)[SODECL_FC][SODE_FIELDS],
                                        const double (&sum)[SODE_FIELDS], const double (&l)[SODECL_FC], sodecl_field_params& pp,
                                        int lane, double (&gx)[SODECL_FC], sodecl_field_params& grad)
{
    double sbar[SODE_FIELDS];
#pragma unroll
    for (int k = 0; k < SODE_FIELDS; ++k) sbar[k] = 0.0;
#pragma unroll
    for (int c = 0; c < SODECL_FC; ++c)   // l is 0 where the component does not exist
        sode_field_vjp_sum(SODECL_FINDEX(c), t, x[c], pp.ps, pp.po[c], const_cast<double*>(phi[c]), const_cast<double*>(sum), l[c],
                           sbar);
    sodecl_field_reduce(sbar);
#pragma unroll
    for (int c = 0; c < SODECL_FC; ++c) {
        const double v = sode_field_vjp(SODECL_FINDEX(c), t, x[c], pp.ps, pp.po[c], const_cast<double*>(phi[c]),
                                        const_cast<double*>(sum), sbar, l[c]);
        gx[c] = SODECL_FOWNS(c) ? v : 0.0;
        sode_field_vjp_params(SODECL_FINDEX(c), t, x[c], pp.ps, pp.po[c], const_cast<double*>(phi[c]), const_cast<double*>(sum),
                              l[c], grad.ps, grad.po[c]);
    }
}

extern "C" __global__ void __launch_bounds__(SODECL_FBLOCK) SODECL_KERNEL_ATTR
sodecl_field_adjoint(const double* __restrict__ ckpt_t, const double* __restrict__ ckpt_y,
                     const double* __restrict__ params, const double* __restrict__ cot,
                     double* __restrict__ grad_y0, double* __restrict__ grad_p, double* __restrict__ work,
                     int orbits, int total_steps, int ckpt_every, int stored)
{
    SODECL_EXP_TABLE_INIT();
    const int lane = sodecl_field_lane(threadIdx.x);
    const int slot = sodecl_field_slot(threadIdx.x);
    const int orbit = blockIdx.x * SODECL_FOPB + slot;
    const bool active = orbit < orbits;
    const int ob = active ? orbit : 0;   // inactive groups read orbit 0's inputs and store nothing
    sodecl_field_params pp;
    sodecl_field_load_params(params + (size_t)ob * _numpar_, true, lane, pp);
    const size_t slab = (size_t)_numeq_ * (size_t)orbits;
    double lam[SODECL_FC];
    // cotangent of the final snapshot (step total_steps)
#pragma unroll
    for (int c = 0; c < SODECL_FC; ++c)
        lam[c] = SODECL_FOWNS(c) ? cot[(size_t)(total_steps / _numsteps_) * slab +
                                       (size_t)(lane * SODECL_FC + c) * orbits + ob]
                                 : 0.0;
    sodecl_field_params grad;
#pragma unroll
    for (int k = 0; k < SODECL_FPS; ++k) grad.ps[k] = 0.0;
#pragma unroll
    for (int c = 0; c < SODECL_FC; ++c)
#pragma unroll
        for (int k = 0; k < SODECL_FPO; ++k) grad.po[c][k] = 0.0;
    // rows of this orbit's segment, read back only by the lanes that wrote
    // them; with stored rows the forward pass wrote every step's
    const size_t rows = (size_t)orbits * (size_t)ckpt_every, row0 = (size_t)ob * (size_t)ckpt_every;
    const int nseg = (total_steps + ckpt_every - 1) / ckpt_every;
    for (int seg = nseg - 1; seg >= 0; --seg) {
        const int sb = seg * ckpt_every;
        const int se = min(total_steps, sb + ckpt_every);
        double y[SODECL_FC];
        double t = 0.0;
        if (!stored) {
#pragma unroll
            for (int c = 0; c < SODECL_FC; ++c)
                y[c] = SODECL_FOWNS(c)
                           ? ckpt_y[(size_t)seg * slab + (size_t)(lane * SODECL_FC + c) * orbits + ob]
                           : 1.0;
            t = ckpt_t[(size_t)seg * orbits + ob];
            for (int s = sb; s < se; ++s) {
                if (active) sodecl_field_store(work, rows, row0 + (s - sb), t, y, lane);
                if (s + 1 < se) {   // the last state needs no successor
                    sodecl_field_step(t, y, pp, lane);
                    t = t + _m_dt_;
                }
            }
        }
        // row of the step ahead, loaded while the step before it (in the sweep) is worked on
        double yn[SODECL_FC], tn = 0.0;
        auto load = [&](int s) {
            const size_t row = row0 + (s - sb);
#pragma unroll
            for (int c = 0; c < SODECL_FC; ++c)
                yn[c] = (active && SODECL_FOWNS(c)) ? work[row * _numeq_ + lane * SODECL_FC + c] : 1.0;
            tn = active ? work[rows * _numeq_ + row] : 0.0;
        };
        if (se > sb) load(se - 1);
        for (int s = se - 1; s >= sb; --s) {
            double phi[SODECL_FSTAGES][SODECL_FC][SODE_FIELDS], sum[SODECL_FSTAGES][SODE_FIELDS];
            double f[SODECL_FC], gv[SODECL_FC];
#pragma unroll
            for (int c = 0; c < SODECL_FC; ++c) y[c] = yn[c];
            const double ts = tn;
            if (s > sb) load(s - 1);
            sodecl_field_eval(ts, y, pp, lane, phi[0], sum[0], f);
#if SODECL_SOLVER == 1
            // y' = y + f(t, y) dt
            double l1[SODECL_FC];
#pragma unroll
            for (int c = 0; c < SODECL_FC; ++c) l1[c] = _m_dt_ * lam[c];
            sodecl_field_product(ts, y, phi[0], sum[0], l1, pp, lane, gv, grad);
#pragma unroll
            for (int c = 0; c < SODECL_FC; ++c) lam[c] = lam[c] + gv[c];
#else
            // y' = y + (k1 + 2 k2 + 2 k3 + k4) dt / 6, k_i = f(t_i, x_i),
            // x2 = y + dt/2 k1, x3 = y + dt/2 k2, x4 = y + dt k3
            double x2[SODECL_FC], x3[SODECL_FC], x4[SODECL_FC];
#pragma unroll
            for (int c = 0; c < SODECL_FC; ++c) x2[c] = y[c] + (_m_dt_ * 0.50) * f[c];
            sodecl_field_eval(ts + 0.50 * _m_dt_, x2, pp, lane, phi[1], sum[1], f);
#pragma unroll
            for (int c = 0; c < SODECL_FC; ++c) x3[c] = y[c] + (_m_dt_ * 0.50) * f[c];
            sodecl_field_eval(ts + 0.50 * _m_dt_, x3, pp, lane, phi[2], sum[2], f);
#pragma unroll
            for (int c = 0; c < SODECL_FC; ++c) x4[c] = y[c] + _m_dt_ * f[c];
            sodecl_field_eval(ts + _m_dt_, x4, pp, lane, phi[3], sum[3], f);
            double l[SODECL_FC];
#pragma unroll
            for (int c = 0; c < SODECL_FC; ++c) l[c] = (_m_dt_ / 6.00) * lam[c];
            double yb[SODECL_FC], kb[SODECL_FC];
            sodecl_field_product(ts + _m_dt_, x4, phi[3], sum[3], l, pp, lane, gv, grad);
#pragma unroll
            for (int c = 0; c < SODECL_FC; ++c) {
                yb[c] = lam[c] + gv[c];
                kb[c] = (2.00 * _m_dt_ / 6.00) * lam[c] + _m_dt_ * gv[c];
            }
            sodecl_field_product(ts + 0.50 * _m_dt_, x3, phi[2], sum[2], kb, pp, lane, gv, grad);
#pragma unroll
            for (int c = 0; c < SODECL_FC; ++c) {
                yb[c] += gv[c];
                kb[c] = (2.00 * _m_dt_ / 6.00) * lam[c] + (_m_dt_ * 0.50) * gv[c];
            }
            sodecl_field_product(ts + 0.50 * _m_dt_, x2, phi[1], sum[1], kb, pp, lane, gv, grad);
#pragma unroll
            for (int c = 0; c < SODECL_FC; ++c) {
                yb[c] += gv[c];
                kb[c] = l[c] + (_m_dt_ * 0.50) * gv[c];
            }
            sodecl_field_product(ts, y, phi[0], sum[0], kb, pp, lane, gv, grad);
#pragma unroll
            for (int c = 0; c < SODECL_FC; ++c) lam[c] = yb[c] + gv[c];
#endif
            // snapshot of step s: add its cotangent
            if (s % _numsteps_ == 0) {
#pragma unroll
                for (int c = 0; c < SODECL_FC; ++c)
                    if (SODECL_FOWNS(c))
                        lam[c] += cot[(size_t)(s / _numsteps_) * slab + (size_t)(lane * SODECL_FC + c) * orbits + ob];
            }
        }
    }
    // the parameters' gradients: zeros first where no component reads a
    // parameter (gathered in LDS, so that each is written once)
    __shared__ double sh_gp[SODECL_FOPB][SODECL_NPAR_ALLOC];
    double* const gp = sh_gp[slot];
    for (int k = lane; k < _numpar_; k += SODECL_FL) gp[k] = 0.0;
    sodecl_wave_sync();   // an orbit's lanes sit in one wavefront
#pragma unroll
    for (int c = 0; c < SODECL_FC; ++c)
        if (SODECL_FOWNS(c))
#pragma unroll
            for (int k = 0; k < SODE_FIELD_OWN; ++k) {
                const unsigned m = (unsigned)sode_field_own_param(lane * SODECL_FC + c, k);
                if (m < _numpar_) gp[m] = grad.po[c][k];
            }
    sodecl_field_reduce(grad.ps);
    if (lane == 0)
#pragma unroll
        for (int k = 0; k < SODE_FIELD_SHARED && k < _numpar_; ++k) gp[k] = grad.ps[k];
    sodecl_wave_sync();
    if (active) {
#pragma unroll
        for (int c = 0; c < SODECL_FC; ++c)
            if (SODECL_FOWNS(c)) grad_y0[(size_t)orbit * _numeq_ + lane * SODECL_FC + c] = lam[c];
        for (int k = lane; k < _numpar_; k += SODECL_FL) grad_p[(size_t)orbit * _numpar_ + k] = gp[k];
    }
}
#endif  // adjoint
#endif  // field form
