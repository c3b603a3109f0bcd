// step_device.h -- device functions shared by the coarse step's kernels
// (kernels.hip, team.hip): scene record, neighbour rows, pair terms, the
// density candidate and the per-particle epilogues of the two passes.
#pragma once

#include "common.h"

namespace sph {

constexpr int kBlock = 256;

inline unsigned blocks_for(uint32_t n, int block) { return (n + block - 1) / block; }

// Scene record of a slot.  ONE (a single scene, every handle's case): index
// 0, a uniform address, so the record's fields are scalar loads; else the
// binary search over the scene begins, per lane (vector loads).
template <bool ONE>
__device__ __forceinline__ const DevScene& scene_for(const DevScene* __restrict__ scenes,
                                                     const uint32_t* __restrict__ begins, int nscenes, uint32_t s) {
    return ONE ? scenes[0] : scenes[scene_of(begins, nscenes, s)];
}

// x^2 + y^2 + z^2 with the contraction written out: two kernels that must
// agree bit for bit cannot leave the choice of the fused product to the
// compiler.
__device__ __forceinline__ float sq3(float x, float y, float z) { return fmaf(z, z, fmaf(x, x, y * y)); }

// Contiguous slot run of the cells [i0, i1] of one x-row (cells of a row
// have consecutive keys, so their particles are consecutive slots).
__device__ __forceinline__ void row_run(const int2* __restrict__ range, uint32_t rowbase, int i0, int i1, int& b,
                                        int& e) {
    b = 0x7fffffff;
    e = -1;
    for (int i = i0; i <= i1; ++i) {
        int2 r = range[rowbase + (uint32_t)i];
        if (r.x >= 0) {
            b = min(b, r.x);
            e = max(e, r.y);
        }
    }
}

// Neighbour range of a particle on the coarse grid (compute_grid_coordinate,
// cu:1238-1258) and the nine x-row runs of it.
struct Rows {
    int lx, hx, ly, hy, lz, hz;
};

__device__ __forceinline__ Rows neighbour_rows(const DevScene& S, float4 xi) {
    const float h = S.h;
    Rows r;
    r.lx = range_coord(xi.x, -h, S.ox, S.cell, S.nx); r.hx = range_coord(xi.x, h, S.ox, S.cell, S.nx);
    r.ly = range_coord(xi.y, -h, S.oy, S.cell, S.ny); r.hy = range_coord(xi.y, h, S.oy, S.cell, S.ny);
    r.lz = range_coord(xi.z, -h, S.oz, S.cell, S.nz); r.hz = range_coord(xi.z, h, S.oz, S.cell, S.nz);
    return r;
}

// Slot run of row (dk, dj) of the 3x3 row set; empty when the row is outside
// the clamped range (e.g. at the grid edge, or the reference's wrapped upper
// coordinate).
__device__ __forceinline__ void row_slots(const int2* __restrict__ range, const DevScene& S, const Rows& R, int dk,
                                          int dj, float4 xi, int& b, int& e) {
    const int k = R.lz + dk, j = R.ly + dj;
    b = 0;
    e = 0;
    if (k > R.hz || j > R.hy) return;
    // a row whose y-z cell rectangle is farther than h from the particle
    // holds no neighbour (its candidates would add exact zeros); the 1e-5
    // margin covers the rounding of the cell bounds and of the keys
    const float y0 = S.oy + (float)j * S.cell, z0 = S.oz + (float)k * S.cell;
    const float dy = fmaxf(fmaxf(y0 - xi.y, xi.y - (y0 + S.cell)), 0.0f);
    const float dz = fmaxf(fmaxf(z0 - xi.z, xi.z - (z0 + S.cell)), 0.0f);
    if (fmaf(dy, dy, dz * dz) * 0.99999f > S.h2) return;
    uint32_t rowbase = S.cell_offset + (uint32_t)(S.nx * (S.ny * k + j));
    row_run(range, rowbase, R.lx, R.hx, b, e);
    if (e < b) { b = 0; e = 0; }
}

// Pair terms of the acceleration (cu:1486-1555) accumulated without the
// constant factors: m, gradSpiky, mu, laplVisc, gradPoly6, laplPoly6 are
// applied once in force_finish.
struct PairSums {
    float fpx, fpy, fpz, fvx, fvy, fvz, cgx, cgy, cgz, cl;
};

// One pair's factors: the vector sums add weight * difference, the colour
// Laplacian iq * lq.
struct PairWeights {
    float cp, wv, wc, iq;                 // pressure, viscosity, colour gradient, colour Laplacian
    float dx, dy, dz, ux, uy, uz, lq;     // x_i - x_j, v_j - v_i, 3 h^2 - 7 r^2
};

// GUARD: the caller has not tested r2 > 0; a pair at distance 0 then adds
// exact zeros (inverse distance and 1/rho_j taken as 0).
template <bool GUARD>
__device__ __forceinline__ PairWeights pair_weights(float4 xi, float4 vi, float rhoi, float Ai, float h, float h2,
                                                    float stiff, float kr0, float4 xj, float4 vj) {
    PairWeights w;
    w.dx = xi.x - xj.x; w.dy = xi.y - xj.y; w.dz = xi.z - xj.z;
    float r2 = sq3(w.dx, w.dy, w.dz);
    float inv_r = __builtin_amdgcn_rsqf(r2);
    float invj = __builtin_amdgcn_rcpf(vj.w);
    if (GUARD) {
        const bool ok = r2 > 0.0f;
        inv_r = ok ? inv_r : 0.0f;
        invj = ok ? invj : 0.0f;
    }
    float rn = r2 * inv_r;
    float pj = stiff * vj.w - kr0;
    float hr = h - rn;
    float qd = h2 - r2;
    w.cp = (Ai + rhoi * pj * invj * invj) * hr * hr * inv_r;
    w.wv = invj * hr;
    w.ux = vj.x - vi.x; w.uy = vj.y - vi.y; w.uz = vj.z - vi.z;
    w.wc = invj * qd * qd;
    w.iq = invj * qd;
    w.lq = 3.0f * h2 - 7.0f * r2;
    return w;
}

template <bool GUARD = false>
__device__ __forceinline__ void pair_terms(PairSums& a, float4 xi, float4 vi, float rhoi, float Ai, float h, float h2,
                                           float stiff, float kr0, float4 xj, float4 vj) {
    const PairWeights w = pair_weights<GUARD>(xi, vi, rhoi, Ai, h, h2, stiff, kr0, xj, vj);
    a.fpx += w.cp * w.dx; a.fpy += w.cp * w.dy; a.fpz += w.cp * w.dz;
    a.fvx += w.wv * w.ux; a.fvy += w.wv * w.uy; a.fvz += w.wv * w.uz;
    a.cgx += w.wc * w.dx; a.cgy += w.wc * w.dy; a.cgz += w.wc * w.dz;
    a.cl += w.iq * w.lq;
}

// Wall penalty + wall viscosity or surface tension (cu:407-466), a = F/rho - g
// (cu:470-473), symplectic Euler (integrate_euler, cu:632-665), the
// grid-driven collision response (collision_handling, cu:742-834) and the
// next step's cell key; writes the next storage order (this step's sorted
// order).
__device__ __forceinline__ void force_finish(const DevScene& S, uint32_t s, float4 xi, float4 vi, const PairSums& a,
                                             const float4* __restrict__ grid4, const float* __restrict__ gridd,
                                             const uint32_t* __restrict__ oid_b, const uint8_t* __restrict__ state_b,
                                             float4* __restrict__ acc, float4* __restrict__ pos_out,
                                             float4* __restrict__ vel_out, uint32_t* __restrict__ oid_out,
                                             uint8_t* __restrict__ state_out, uint32_t* __restrict__ key_out,
                                             uint32_t* __restrict__ status, const NeuralRefs& nr, bool by_id = false) {
    const float rhoi = vi.w;
    const float cpf = -S.mass * S.grad_spiky, cvf = S.mu * S.mass * S.lapl_visc;
    float Fx = fmaf(cvf, a.fvx, cpf * a.fpx), Fy = fmaf(cvf, a.fvy, cpf * a.fpy), Fz = fmaf(cvf, a.fvz, cpf * a.fpz);
    const int wm = wall_mode(nr, s);
    float tx, ty, tz;
    texel_coords(S, xi.x, xi.y, xi.z, tx, ty, tz);
    // distance and wall viscosity from the grid (the wall-term switch
    // distWall < r0 and the penalty magnitude need its exact values); a cell
    // far from every surface takes no wall term and no lookup; with the
    // learned source the penalty and collision normals come from the
    // network's gradient instead of central differences of the grid
    float distWall = S.r0, wvisc = 0.0f;
    float4 r1 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (wm != kWallNone) {
        float4 g = lerp3<float4>(grid4, S, tex_setup(S, tx, ty, tz));
        distWall = -g.x;
        wvisc = g.z;
        if (wm == kWallNeural && nr.need[s]) r1 = nr.rec[s];   // central-difference gradient of the learned distance at x
    }
    // the network's normal exists where the density pass asked for it
    const bool net_normal = wm == kWallNeural && nr.need[s];
    if (distWall < S.r0) {
        float coeff = rhoi / (S.dt * S.dt) * (S.r0 - distWall);
        // normalized-coordinate gradient: learned source dD/dx times
        // dx/du = L = dims / bscale per axis
        float3 gn = net_normal ? make_float3(r1.x * ((float)S.bnx / S.bscale_x), r1.y * ((float)S.bny / S.bscale_y),
                                             r1.z * ((float)S.bnz / S.bscale_z))
                               : dist_grad_normalized(gridd, S, tx, ty, tz);
        Fx -= fmaf(coeff, gn.x, vi.x * wvisc);
        Fy -= fmaf(coeff, gn.y, vi.y * wvisc);
        Fz -= fmaf(coeff, gn.z, vi.z * wvisc);
    } else {
        float cm = S.mass * S.grad_poly6;
        float gx = cm * a.cgx, gy = cm * a.cgy, gz = cm * a.cgz;
        float gnorm = sqrtf(sq3(gx, gy, gz));
        if (gnorm > S.norm_thresh) {
            float fc = S.sigma * (S.mass * S.lapl_poly6 * a.cl) / gnorm;
            Fx -= fc * gx;
            Fy -= fc * gy;
            Fz -= fc * gz;
        }
    }
    float ax = Fx / rhoi, ay = Fy / rhoi - S.gravity, az = Fz / rhoi;
    acc[s] = make_float4(ax, ay, az, 0.0f);
    float vx = vi.x + S.dt * ax, vy = vi.y + S.dt * ay, vz = vi.z + S.dt * az;
    float px = xi.x + S.dt * vx, py = xi.y + S.dt * vy, pz = xi.z + S.dt * vz;
    if (S.collision && wm != kWallNone) {
        float D;
        float3 gw;
        float cx, cy, cz;
        texel_coords(S, px, py, pz, cx, cy, cz);
        D = dist_at(gridd, S, cx, cy, cz);
        if (D > 0.0f) {
            if (net_normal) {
                gw = make_float3(r1.x, r1.y, r1.z);   // learned source: its gradient at the old position
            } else {
                gw = dist_grad_normalized(gridd, S, cx, cy, cz);
                // normalized-coordinate gradient -> world gradient: divide by L
                gw.x *= S.bscale_x * (1.0f / (float)S.bnx);
                gw.y *= S.bscale_y * (1.0f / (float)S.bny);
                gw.z *= S.bscale_z * (1.0f / (float)S.bnz);
            }
        }
        if (D > 0.0f) {
            float gl = sqrtf(sq3(gw.x, gw.y, gw.z));
            if (gl > 0.0f) {
                float nx_ = gw.x / gl, ny_ = gw.y / gl, nz_ = gw.z / gl;
                float vn = sqrtf(sq3(vx, vy, vz));
                float dp = fmaf(nz_, vz, fmaf(nx_, vx, ny_ * vy));
                float c = 1.0f;
                if (S.restitution != 0.0f && vn > 0.0f) c += S.restitution * D / (S.dt * vn);
                c *= dp;
                vx -= c * nx_; vy -= c * ny_; vz -= c * nz_;
                px -= D * nx_; py -= D * ny_; pz -= D * nz_;
            }
        }
    }
    uint32_t flags = 0;
    uint32_t kk = cell_key(S, px, py, pz, flags);
    if (!(isfinite(px) && isfinite(py) && isfinite(pz) && isfinite(vx) && isfinite(vy) && isfinite(vz)))
        flags |= kStatusNonFinite;
    if (flags) atomicOr(status, flags);
    const uint32_t id = oid_b[s], at = by_id ? id : s;
    pos_out[at] = make_float4(px, py, pz, rhoi);
    vel_out[at] = make_float4(vx, vy, vz, rhoi);
    key_out[s] = kk;
    oid_out[s] = id;
    if (state_out) state_out[s] = state_b[s];
}

__device__ __forceinline__ float wall_density(const DevScene& S, const float4* __restrict__ grid4, float4 xi,
                                              const NeuralRefs& nr, uint32_t s) {
    // the density pass flags the network's particles; it also starts their
    // lists (the network pass appends after it)
    if (s == 0 && nr.list_count)
        for (int i = 0; i < nr.nscenes; ++i) nr.list_count[i] = 0u;
    const int wm = wall_mode(nr, s);
    if (wm == kWallNone) return 0.0f;
    float tx, ty, tz;
    texel_coords(S, xi.x, xi.y, xi.z, tx, ty, tz);
    const float4 g = lerp3<float4>(grid4, S, tex_setup(S, tx, ty, tz));
    // learned source: the force pass needs the network's normal exactly
    // where the wall penalty acts (distWall = -D < r0)
    if (wm == kWallNeural && nr.need) nr.need[s] = g.x > -S.r0;
    return g.y;
}

// h^2 - r^2 of a candidate, clamped at 0, as the variants without masks form
// it (their poly6 term is its cube).
__device__ __forceinline__ float density_gap(float4 xi, float4 xj, float h2) {
    float dx = xj.x - xi.x, dy = xj.y - xi.y, dz = xj.z - xi.z;
    return fmaxf(h2 - sq3(dx, dy, dz), 0.0f);
}

// One candidate of the density pass: poly6 sum and the "farther than h" bit.
// d = h2 - dz^2 - dy^2 - dx^2 as a chain of three fused multiply-adds (one
// instruction fewer than forming r^2 and subtracting it).  Each step rounds
// an exact result, which keeps its sign (and an exact zero is +0), so d's
// sign bit is set exactly when this d is negative, i.e. when the candidate's
// poly6 term is zero: the bit is that "farther than h" bit and one funnel
// shift per candidate builds the mask.  GAP: the d of density_gap instead, and
// the bit is exactly !(0 < r^2 <= h^2), the test of the loops without masks,
// whatever the values (three instructions more).
template <bool GAP = false>
__device__ __forceinline__ void density_candidate(float xjx, float xjy, float xjz, float4 xi, float h2, float& sum,
                                                  uint32_t& far) {
    float dx = xjx - xi.x, dy = xjy - xi.y, dz = xjz - xi.z;
    float d, bit;
    if (GAP) {
        const float r2 = sq3(dx, dy, dz);
        d = h2 - r2;
        bit = r2 > 0.0f ? d : -1.0f;
    } else {
        bit = d = fmaf(-dx, dx, fmaf(-dy, dy, fmaf(-dz, dz, h2)));
    }
    far = __builtin_amdgcn_alignbit(far, __float_as_uint(bit), 31);
    d = fmaxf(d, 0.0f);
    sum += d * d * d;
}

}  // namespace sph
