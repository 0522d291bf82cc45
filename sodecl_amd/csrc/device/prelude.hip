// Device helpers visible to the system plugin (emitted before it).

// A double moved across lanes by one DPP control (two 32-bit moves); a lane
// whose source lies outside its row or the wavefront, or is not active,
// receives 0 (the instruction's own bound control: no register has to hold
// the 0 beforehand, which cost a move per 32-bit half).
template <int CTRL>
__device__ inline double sodecl_dpp(double v)
{
    const long long bits = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_mov_dpp((int)(bits & 0xffffffffll), CTRL, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_mov_dpp((int)(bits >> 32), CTRL, 0xF, 0xF, true);
    return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned int)lo);
}
#define SODECL_DPP_XOR1 0xB1          // quad_perm [1,0,3,2]
#define SODECL_DPP_XOR2 0x4E          // quad_perm [2,3,0,1]
#define SODECL_DPP_XOR3 0x1B          // quad_perm [3,2,1,0]
#define SODECL_DPP_HALF_MIRROR 0x141  // lane i <- 7 - i within each 8 lanes
#define SODECL_DPP_MIRROR 0x140       // lane i <- 15 - i within each 16 lanes
#define SODECL_DPP_WAVE_SHR1 0x138    // lane i <- lane i - 1 across the wavefront (lane 0 <- 0)
#define SODECL_DPP_WAVE_SHL1 0x130    // lane i <- lane i + 1 across the wavefront (lane 63 <- 0)
#define SODECL_DPP_ROW_SHR(n) (0x110 + (n))   // lane i <- lane i - n within its 16-lane row (0 past the start)
#define SODECL_DPP_ROW_SHL(n) (0x100 + (n))   // lane i <- lane i + n within its 16-lane row (0 past the end)

// 1/b from the hardware reciprocal r (relative error e = 1 - b r, below 2^-20)
// and one step of third order, r + r (e + e^2), which leaves e^3 and the last
// rounding (within an ulp, for solves that are not the reference's operation by
// operation; one instruction less than two Newton-Raphson steps, and issue
// bounds those solves).
__device__ inline double sodecl_rcp(double b)
{
    const double r = __builtin_amdgcn_rcp(b);
    const double e = fma(-b, r, 1.0);
    return fma(r, fma(e, e, e), r);
}

// A value known to be a zero when the kernel is compiled: a coefficient the
// plugin gives as a constant zero.  Its products drop out of an elimination or
// a sum (they would be zeros added to finite values).
__device__ __attribute__((always_inline)) inline bool sodecl_zero(double v)
{
    return __builtin_constant_p(v) && v == 0.0;
}

// Orders this wavefront's LDS accesses before the call against those after
// it, for exchanges among the lanes of one wavefront: DS instructions of one
// wavefront execute in order, and the fences plus the wave barrier keep the
// compiler from moving LDS accesses across this point.  No other wavefront
// is waited for.
__device__ inline void sodecl_wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Under the group schedule SODECL_GROUP consecutive lanes of a wavefront
// share one orbit.  A plugin entry point that the whole group calls together
// (sode_system_vjp_group) may use:
//   sodecl_group_size()  lanes per orbit
//   sodecl_lane()        this lane's index within the group, 0..G-1
//   sodecl_group_sum(v)  sum of v over the group, the same value on every lane
// These exist only in device code compiled for the group schedule
// (SODECL_GROUP_API is defined there).
#if SODECL_SCHEDULE == 2
__device__ inline int sodecl_group_size() { return SODECL_GROUP; }
__device__ inline int sodecl_lane() { return (int)(threadIdx.x % SODECL_GROUP); }
// Reduction over aligned blocks of W lanes in levels of lane distance 1, 2,
// 4, 8, 16, 32.  The first four are DPP moves inside a 16-lane row: xor 1 and
// xor 2 by quad permutations, then the half-row and row mirrors, which pair
// every lane with the opposite block of the previous level (whose lanes all
// hold the same partial sum) exactly as xor 4 and xor 8 would.  The last two
// swap rows (v_permlane16_swap) or half wavefronts (v_permlane32_swap) of two
// copies of the value, one register per 32-bit half: the copies then hold one
// partner's sum each on both partners.  At every level the two partners add
// the same two numbers, so every lane ends with a bit-identical sum.
__device__ inline double sodecl_swapped_sum(double v, bool rows)
{
    const long long bits = __double_as_longlong(v);
    const int l = (int)(bits & 0xffffffffll), h = (int)(bits >> 32);
    const auto lo = rows ? __builtin_amdgcn_permlane16_swap(l, l, false, false)
                         : __builtin_amdgcn_permlane32_swap(l, l, false, false);
    const auto hi = rows ? __builtin_amdgcn_permlane16_swap(h, h, false, false)
                         : __builtin_amdgcn_permlane32_swap(h, h, false, false);
    return __longlong_as_double(((long long)(int)hi[0] << 32) | (long long)(unsigned int)lo[0]) +
           __longlong_as_double(((long long)(int)hi[1] << 32) | (long long)(unsigned int)lo[1]);
}
// Several sums at once, level by level.
template <int W, int K>
__device__ inline void sodecl_lane_sums(double (&v)[K])
{
#define SODECL_LANE_LEVEL(LANES, SUM)                             \
    if (W >= LANES)                                               \
        _Pragma("unroll") for (int k = 0; k < K; ++k) v[k] = SUM;
    SODECL_LANE_LEVEL(2, v[k] + sodecl_dpp<SODECL_DPP_XOR1>(v[k]))
    SODECL_LANE_LEVEL(4, v[k] + sodecl_dpp<SODECL_DPP_XOR2>(v[k]))
    SODECL_LANE_LEVEL(8, v[k] + sodecl_dpp<SODECL_DPP_HALF_MIRROR>(v[k]))
    SODECL_LANE_LEVEL(16, v[k] + sodecl_dpp<SODECL_DPP_MIRROR>(v[k]))
    SODECL_LANE_LEVEL(32, sodecl_swapped_sum(v[k], true))
    SODECL_LANE_LEVEL(64, sodecl_swapped_sum(v[k], false))
#undef SODECL_LANE_LEVEL
}
__device__ inline double sodecl_group_sum(double v)
{
    double s[1] = {v};
    sodecl_lane_sums<SODECL_GROUP>(s);
    return s[0];
}
#define SODECL_GROUP_API 1
#endif

// Under the team schedule SODECL_GROUP consecutive lanes share one orbit and
// every one of them holds the whole state.  The plugin's team entry point
// (sode_system_team), called by all lanes of the team together with the same
// arguments, may split the drift among them and must return it complete on
// every lane.  It may use:
//   sodecl_group_size()     lanes per orbit
//   sodecl_lane()           this lane's index within the team, 0..G-1
//   sodecl_group_xor(v, m)  v of team lane sodecl_lane() ^ m (m < G)
// These exist only in device code compiled for the team schedule, and for
// Euler-Maruyama launches of the lane schedule whose orbits have several lanes
// (SODECL_TEAM_API is defined there).  The lanes of such an orbit are teams of
// two, as in an automatic team launch: a source may be written for pairs.
#if SODECL_SCHEDULE == 4
#define SODECL_TEAM_LANES SODECL_GROUP
#elif SODECL_SCHEDULE == 1 && defined(SODECL_NOISE_TEAM)
#define SODECL_TEAM_LANES 2
#endif
#ifdef SODECL_TEAM_LANES
__device__ inline int sodecl_group_size() { return SODECL_TEAM_LANES; }
__device__ inline int sodecl_lane() { return (int)(threadIdx.x % SODECL_TEAM_LANES); }
// Lane exchange within quads by DPP quad permutations for m = 1, 2, 3
// (no LDS traffic), cross-lane permute otherwise.
__device__ inline double sodecl_group_xor(double v, int m)
{
    switch (m) {
    case 1: return sodecl_dpp<SODECL_DPP_XOR1>(v);
    case 2: return sodecl_dpp<SODECL_DPP_XOR2>(v);
    case 3: return sodecl_dpp<SODECL_DPP_XOR3>(v);
    default: return __shfl_xor(v, m, SODECL_TEAM_LANES);
    }
}
#define SODECL_TEAM_API 1
#endif
