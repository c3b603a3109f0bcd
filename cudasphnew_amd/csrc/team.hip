// team.hip -- the density and force passes for small particle sets: sixteen
// lanes ("a team") share one particle.
//
// With one thread per particle a set of a few thousand particles is a
// handful of wavefronts, and a pass lasts as long as one wavefront's chain
// of dependent loads (nine rows, each a cell-table read followed by batches
// of candidate reads): 22 us (density) and 35 us (force) from 700 to 16,384
// particles.  A team reads its nine rows' cell ranges in one round and 16
// candidates of a row per load, every row's loads in flight together, so a
// pass is a few round trips, on 16 times as many wavefronts.  Measured, per
// launch: density 22 -> 6 us and force 35 -> 10 us at 700 particles, 23 -> 13
// and 36 -> 16 us at 16,384.
//
// The results are those of the one-thread kernels bit for bit: a particle's
// terms are evaluated in parallel, written to LDS in candidate order and
// summed serially in that order (a far candidate adds an exact zero and is
// left out), so which kernel a set takes -- alone, in a batch, through
// sph_step_noalloc -- does not show in its results.
#include "kernels.h"
#include "step_device.h"

namespace sph {

namespace {

constexpr int kTeam = 16;                    // lanes per particle
constexpr int kTeams = kBlock / kTeam;       // particles per workgroup
constexpr int kRow = 32;                     // candidates of a row on the fast path
constexpr int kList = 9 * kRow;              // list entries per team: every candidate of the fast path
constexpr int kPad = kList + kTeam;          // + the zero padding of a partial vector read

// The nine rows' runs of a team's particle: lane r < 9 finds row r, then all
// lanes hold all rows.  b and cnt are indexed with constants only (a loop
// over them that stays a loop puts both in scratch memory); row(r) asks lane r.
struct TeamRows {
    int b[9], cnt[9];
    int own_b, own_cnt;
    __device__ __forceinline__ void row(int r, int& rb, int& rcnt) const {
        rb = __shfl(own_b, r, kTeam);
        rcnt = __shfl(own_cnt, r, kTeam);
    }
};

__device__ __forceinline__ TeamRows team_rows(const int2* __restrict__ range, const DevScene& S, float4 xi, int c) {
    const Rows R = neighbour_rows(S, xi);
    int b = 0, e = 0;
    if (c < 9) row_slots(range, S, R, c / 3, c % 3, xi, b, e);
    TeamRows t;
    t.own_b = b;
    t.own_cnt = e - b;
#pragma unroll
    for (int r = 0; r < 9; ++r) {
        t.b[r] = __shfl(b, r, kTeam);
        t.cnt[r] = __shfl(t.own_cnt, r, kTeam);
    }
    return t;
}

// Which candidates are neighbours, as the kernel pair replaced here decides
// it.  MASKS: the hit-mask pair (sign of h^2 - r^2 in three fused steps, the
// own slot left out; a distinct particle at distance 0 stays and adds
// zeros); else r^2 <= h^2 and r^2 > 0.
template <bool MASKS>
__device__ __forceinline__ bool is_neighbour(float4 xi, float4 xj, float h2, bool self) {
    if (MASKS) {
        const float dx = xj.x - xi.x, dy = xj.y - xi.y, dz = xj.z - xi.z;
        const float d = fmaf(-dx, dx, fmaf(-dy, dy, fmaf(-dz, dz, h2)));
        return !(__float_as_uint(d) >> 31) && !self;
    }
    const float dx = xi.x - xj.x, dy = xi.y - xj.y, dz = xi.z - xj.z;
    const float r2 = sq3(dx, dy, dz);
    return r2 <= h2 && r2 > 0.0f;
}

// Clamped h^2 - r^2 of a candidate in the replaced kernel's arithmetic.
template <bool MASKS>
__device__ __forceinline__ float team_gap(float4 xi, float4 xj, float h2) {
    if (!MASKS) return density_gap(xi, xj, h2);
    const float dx = xj.x - xi.x, dy = xj.y - xi.y, dz = xj.z - xi.z;
    return fmaxf(fmaf(-dx, dx, fmaf(-dy, dy, fmaf(-dz, dz, h2))), 0.0f);
}

// Appends `value` of the lanes with `take` to the team's list in lane order;
// returns the new length.
template <class T>
__device__ __forceinline__ int team_append(T* list, int m, bool take, T value, int c, int shift) {
    const uint32_t bits = (uint32_t)(__ballot(take) >> shift) & 0xFFFFu;
    if (take) list[m + __popc(bits & ((1u << c) - 1u))] = value;
    return m + __popc(bits);
}

// Adds the cubes of list[0, m) to sum, in order (every lane of the team).
__device__ __forceinline__ float sum_cubes(float* list, int m, float sum, int c) {
    list[m + c] = 0.0f;   // a partial vector of four adds zeros
    wave_sync();
    for (int k = 0; k < m; k += 4) {
        const float4 d = *reinterpret_cast<const float4*>(list + k);
        sum += d.x * d.x * d.x;
        sum += d.y * d.y * d.y;
        sum += d.z * d.z * d.z;
        sum += d.w * d.w * d.w;
    }
    wave_sync();
    return sum;
}

template <bool MASKS, bool ONE>
__global__ __launch_bounds__(kBlock) void k_density_team(const float4* __restrict__ pos, float4* __restrict__ vel,
                                                         const int2* __restrict__ range, uint32_t n,
                                                         const DevScene* __restrict__ scenes,
                                                         const uint32_t* __restrict__ begins, int nscenes,
                                                         const float4* __restrict__ grid4, NeuralRefs nr) {
    __shared__ __align__(16) float s_list[kTeams][kPad];
    const int c = threadIdx.x % kTeam;
    const int shift = (threadIdx.x & 63) / kTeam * kTeam;
    float* list = s_list[threadIdx.x / kTeam];
    const uint32_t s0 = xcd_block(blockIdx.x, gridDim.x) * kTeams + threadIdx.x / kTeam;
    const bool live = s0 < n;                  // the teams past the end repeat the last particle
    const uint32_t s = live ? s0 : n - 1;
    const DevScene& S = scene_for<ONE>(scenes, begins, nscenes, s);
    const float4 xi = pos[s];
    const float h2 = S.h2;
    const TeamRows T = team_rows(range, S, xi, c);
    int longest = 0;
#pragma unroll
    for (int r = 0; r < 9; ++r) longest = max(longest, T.cnt[r]);
    float sum = 0.0f;
    int m = 0;
    if (__all(longest <= kRow)) {
        float gap[18];
#pragma unroll
        for (int r = 0; r < 9; ++r)
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int t = kTeam * u + c;
                const bool in = t < T.cnt[r];
                const float4 xj = pos[in ? (uint32_t)(T.b[r] + t) : s];
                const float d = team_gap<MASKS>(xi, xj, h2);
                gap[2 * r + u] = in ? d : 0.0f;
            }
#pragma unroll
        for (int k = 0; k < 18; ++k) m = team_append(list, m, gap[k] > 0.0f, gap[k], c, shift);
    } else {
        // longer rows (a compressed flow): the list is summed whenever another
        // 16 might not fit
#pragma unroll 1
        for (int r = 0; r < 9; ++r) {
            int b, cnt;
            T.row(r, b, cnt);
            for (int t0 = 0; __any(t0 < cnt); t0 += kTeam) {
                const bool in = t0 + c < cnt;
                const float4 xj = pos[in ? (uint32_t)(b + t0 + c) : s];
                const float d = team_gap<MASKS>(xi, xj, h2);
                m = team_append(list, m, in && d > 0.0f, d, c, shift);
                if (__any(m > kList - kTeam)) {
                    sum = sum_cubes(list, m, sum, c);
                    m = 0;
                }
            }
        }
    }
    sum = sum_cubes(list, m, sum, c);
    if (c == 0 && live) {
        const float rho = sum * (S.poly6 * S.mass) + wall_density(S, grid4, xi, nr, s);
        reinterpret_cast<float*>(vel)[4 * (size_t)s + 3] = rho;
    }
}

// LDS of a wavefront's pair factors: row f holds factor f of the 64 lanes'
// pairs, a multiple of four floats apart with the rows on different banks.
constexpr int kTermStride = 68;

// Sums of a team, one component per lane: lane c < 9 owns fp, fv, cg (x, y,
// z each), lane 9 the colour Laplacian.  Adds the pairs of list[0, m) in
// order.
template <bool MASKS>
__device__ __forceinline__ float team_pairs(const float4* __restrict__ pos, const float4* __restrict__ vel,
                                            const int* list, int m, float* terms, const DevScene& S, float4 xi,
                                            float4 vi, uint32_t s, int c, int shift, float acc) {
    const float h = S.h, h2 = S.h2, rhoi = vi.w;
    const float Ai = S.stiff * (rhoi - S.rho0) / rhoi;   // p_i / rho_i
    const float kr0 = S.stiff * S.rho0;
    const int row_a = c < 9 ? c / 3 : 3;
    const int row_b = c < 3 ? 4 + c : (c < 6 ? 4 + c : (c < 9 ? c - 2 : 10));
    const float* ta = terms + row_a * kTermStride + shift;
    const float* tb = terms + row_b * kTermStride + shift;
    float* mine = terms + shift + c;
    uint32_t q = c < m ? (uint32_t)list[c] : s;
    float4 xj = pos[q], vj = vel[q];
    for (int k0 = 0; __any(k0 < m); k0 += kTeam) {
        const bool in = k0 + c < m;
        const PairWeights w = pair_weights<MASKS>(xi, vi, rhoi, Ai, h, h2, S.stiff, kr0, xj, vj);
        // the next round's gathers run while this one is summed
        q = k0 + kTeam + c < m ? (uint32_t)list[k0 + kTeam + c] : s;
        xj = pos[q];
        vj = vel[q];
        mine[0 * kTermStride] = in ? w.cp : 0.0f;
        mine[1 * kTermStride] = in ? w.wv : 0.0f;
        mine[2 * kTermStride] = in ? w.wc : 0.0f;
        mine[3 * kTermStride] = in ? w.iq : 0.0f;
        mine[4 * kTermStride] = in ? w.dx : 0.0f;
        mine[5 * kTermStride] = in ? w.dy : 0.0f;
        mine[6 * kTermStride] = in ? w.dz : 0.0f;
        mine[7 * kTermStride] = in ? w.ux : 0.0f;
        mine[8 * kTermStride] = in ? w.uy : 0.0f;
        mine[9 * kTermStride] = in ? w.uz : 0.0f;
        mine[10 * kTermStride] = in ? w.lq : 0.0f;
        wave_sync();
#pragma unroll
        for (int i = 0; i < kTeam; i += 4) {
            const float4 a = *reinterpret_cast<const float4*>(ta + i);
            const float4 b = *reinterpret_cast<const float4*>(tb + i);
            acc += a.x * b.x;
            acc += a.y * b.y;
            acc += a.z * b.z;
            acc += a.w * b.w;
        }
        wave_sync();
    }
    return acc;
}

template <bool MASKS, bool ONE>
__global__ __launch_bounds__(kBlock) void k_force_team(
    const float4* __restrict__ pos, const float4* __restrict__ vel, const int2* __restrict__ range, uint32_t n,
    const DevScene* __restrict__ scenes, const uint32_t* __restrict__ begins, int nscenes,
    const float4* __restrict__ grid4, const float* __restrict__ gridd, const uint32_t* __restrict__ oid_b,
    const uint8_t* __restrict__ state_b, float4* __restrict__ acc, float4* __restrict__ pos_out,
    float4* __restrict__ vel_out, uint32_t* __restrict__ oid_out, uint8_t* __restrict__ state_out,
    uint32_t* __restrict__ key_out, uint32_t* __restrict__ status, NeuralRefs nr, bool by_id) {
    __shared__ int s_list[kTeams][kList];
    __shared__ __align__(16) float s_terms[kBlock / 64][11 * kTermStride];
    __shared__ float s_sum[10][kTeams];
    const int c = threadIdx.x % kTeam, team = threadIdx.x / kTeam;
    const int shift = (threadIdx.x & 63) / kTeam * kTeam;
    int* list = s_list[team];
    float* terms = s_terms[threadIdx.x >> 6];
    const uint32_t P0 = xcd_block(blockIdx.x, gridDim.x) * kTeams;
    const uint32_t s = min(P0 + (uint32_t)team, n - 1);   // the teams past the end repeat the last particle
    {
        const DevScene& S = scene_for<ONE>(scenes, begins, nscenes, s);
        const float4 xi = pos[s];
        const float4 vi = vel[s];
        const float h2 = S.h2;
        const TeamRows T = team_rows(range, S, xi, c);
        int longest = 0;
#pragma unroll
        for (int r = 0; r < 9; ++r) longest = max(longest, T.cnt[r]);
        float sum = 0.0f;
        int m = 0;
        if (__all(longest <= kRow)) {
            uint32_t near = 0;   // bit 2r + u: this lane's candidate of batch u of row r
#pragma unroll
            for (int r = 0; r < 9; ++r)
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const int t = kTeam * u + c;
                    const bool in = t < T.cnt[r];
                    const uint32_t q = in ? (uint32_t)(T.b[r] + t) : s;
                    const bool hit = in && is_neighbour<MASKS>(xi, pos[q], h2, q == s);
                    near |= (uint32_t)hit << (2 * r + u);
                }
#pragma unroll
            for (int k = 0; k < 18; ++k)
                m = team_append(list, m, (near >> k & 1u) != 0, T.b[k / 2] + kTeam * (k & 1) + c, c, shift);
        } else {
            // the hit-mask pair takes its rows of more than kRowMaxCands
            // candidates after the others, by the plain test
#pragma unroll 1
            for (int k = 0; k < (MASKS ? 18 : 9); ++k) {
                const int r = k % 9;
                const bool late = k >= 9;
                int b, cnt;
                T.row(r, b, cnt);
                if (MASKS && late != (cnt > kRowMaxCands)) cnt = 0;
                for (int t0 = 0; __any(t0 < cnt); t0 += kTeam) {
                    const bool in = t0 + c < cnt;
                    const uint32_t q = in ? (uint32_t)(b + t0 + c) : s;
                    const float4 xj = pos[q];
                    const bool hit = in && (late ? is_neighbour<false>(xi, xj, h2, q == s)
                                                 : is_neighbour<MASKS>(xi, xj, h2, q == s));
                    m = team_append(list, m, hit, (int)q, c, shift);
                    if (__any(m > kList - kTeam)) {
                        wave_sync();
                        sum = team_pairs<MASKS>(pos, vel, list, m, terms, S, xi, vi, s, c, shift, sum);
                        m = 0;
                    }
                }
            }
        }
        wave_sync();
        sum = team_pairs<MASKS>(pos, vel, list, m, terms, S, xi, vi, s, c, shift, sum);
        if (c < 10) s_sum[c][team] = sum;
    }
    __syncthreads();
    // the epilogue: one thread per particle of the workgroup
    const uint32_t p = P0 + threadIdx.x;
    if (threadIdx.x >= kTeams || p >= n) return;
    const DevScene& S = scene_for<ONE>(scenes, begins, nscenes, p);
    PairSums a;
    float* av = &a.fpx;
#pragma unroll
    for (int t = 0; t < 10; ++t) av[t] = s_sum[t][threadIdx.x];
    force_finish(S, p, pos[p], vel[p], a, grid4, gridd, oid_b, state_b, acc, pos_out, vel_out, oid_out, state_out,
                 key_out, status, nr, by_id);
}

unsigned team_blocks(uint32_t n) { return (n + kTeams - 1) / kTeams; }

template <bool MASKS, bool ONE>
void density_team(hipStream_t st, const StepBuffers& b) {
    hipLaunchKernelGGL((k_density_team<MASKS, ONE>), dim3(team_blocks(b.n)), dim3(kBlock), 0, st, b.pos_b, b.vel_b,
                       b.range, b.n, b.scenes, b.begins, b.nscenes, b.grid4, b.nr);
}

template <bool MASKS, bool ONE>
void force_team(hipStream_t st, const StepBuffers& b) {
    hipLaunchKernelGGL((k_force_team<MASKS, ONE>), dim3(team_blocks(b.n)), dim3(kBlock), 0, st, b.pos_b, b.vel_b,
                       b.range, b.n, b.scenes, b.begins, b.nscenes, b.grid4, b.gridd, b.oid_b, b.state_b, b.acc,
                       b.pos_a, b.vel_a, b.oid_a, b.state_a, b.key, b.status, b.nr, b.by_id);
}

// Teams issue about four times the instructions of one thread per particle,
// so they win until the chip is full of wavefronts.  Against the one-lane
// loops, us a step with the sort: 35 / 78 at 4,000 particles, 46 / 78 at 16,384,
// 64 / 79 at 32,768, 85 / 77 at 50,000 (twice rest density: 132 / 141 there);
// against the masks pair, two steps and a read of the positions: 107 / 119 at
// 20,000, 117 / 119 at 25,000, 122 / 120 at 30,000 (twice rest density 146 /
// 187, 160 / 189, 175 / 193).  A two-scale step needs the hit-mask density
// pass's row words and split flags.
constexpr uint32_t kTeamMax = 40960, kTeamMaxMasks = 28672;

}  // namespace

bool team_size(uint32_t n, bool masks) { return n <= (masks ? kTeamMaxMasks : kTeamMax); }

bool team_step(const StepBuffers& b) { return b.teams && team_size(b.n, b.masks != nullptr); }

void launch_density_team(hipStream_t st, const StepBuffers& b) {
    const bool one = b.nscenes == 1;
    if (b.masks) one ? density_team<true, true>(st, b) : density_team<true, false>(st, b);
    else one ? density_team<false, true>(st, b) : density_team<false, false>(st, b);
}

void launch_force_team(hipStream_t st, const StepBuffers& b) {
    const bool one = b.nscenes == 1;
    if (b.masks) one ? force_team<true, true>(st, b) : force_team<true, false>(st, b);
    else one ? force_team<false, true>(st, b) : force_team<false, false>(st, b);
}

}  // namespace sph
