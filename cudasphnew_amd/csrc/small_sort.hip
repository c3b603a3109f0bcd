// small_sort.hip -- the cell sort of a small particle set in one workgroup.
//
// For some thousand particles the counting sort's four launches and the
// reorder pass are bound by launching (2 to 5 us each, whatever they do).  One
// workgroup of 1,024 threads holds the whole count array (16 bits a cell) and
// the particles' ids in LDS and goes through the same steps between barriers:
//   count    each particle's arrival rank in its cell, one LDS atomic
//   scan     cell starts; range of every cell, empty ones included (the table
//            need not be cleared between steps)
//   rank     each particle's rank by original id among its cell's, from LDS
//   place    sorted keys and the sorted copies
// The sorted order is that of CellSort + k_reorder.  Bound by the chain of
// LDS and memory latencies of four particles a thread: 5.9 us for 700
// particles on a 32 x 32 x 32 grid.  One call without a handle (sort,
// density, force) against the four launches: 27.8 and 41.4 us with 1,024
// particles, 35.8 and 42.0 with 4,096 in cell order, 44.0 and 47.2 shuffled.
// Eight particles a thread lose to the launches: 8,192 take 50.5 and 45.4,
// shuffled 66.1 and 48.7 us -- one CU is then the bound of moving 64 bytes a
// particle -- hence the line at 4,096.
#include "kernels.h"
#include "step_device.h"

namespace sph {

namespace {

constexpr int kT = 1024;                // threads
constexpr int kPer = 4;                 // particles a thread
constexpr uint32_t kMaxCells = 48128;   // 94 KiB of counts beside 16 KiB of ids
constexpr int kWords = (int)kMaxCells / 2;

__device__ __forceinline__ uint32_t half_of(const uint32_t* w, uint32_t c) { return w[c >> 1] >> (16 * (c & 1)) & 0xFFFFu; }

// Exclusive scan of one value per thread of the workgroup.
__device__ __forceinline__ uint32_t scan_block(uint32_t v, uint32_t* s_wave) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
    if (lane == 63) s_wave[wave] = x;
    __syncthreads();
    uint32_t off = 0;
#pragma unroll
    for (int w = 0; w < kT / 64; ++w) off += w < wave ? s_wave[w] : 0u;
    return off + x - v;
}

// first.scene != null: the first step of a call
// without a handle -- keys from the positions with S, ids the indices, and
// the call's scene record, slot range and status word written here.
__global__ __launch_bounds__(kT) void k_small_sort(DevScene S, SmallFirst first, const uint32_t* __restrict__ key,
                                                   const uint32_t* __restrict__ oid_a,
                                                   const float4* __restrict__ pos_a, const float4* __restrict__ vel_a,
                                                   const uint8_t* __restrict__ state_a, uint32_t n, uint32_t cells,
                                                   int2* __restrict__ range, uint32_t* __restrict__ skey,
                                                   float4* __restrict__ pos_b, float4* __restrict__ vel_b,
                                                   uint32_t* __restrict__ oid_b, uint8_t* __restrict__ state_b,
                                                   uint32_t* __restrict__ slot_of_oid) {
    __shared__ uint32_t s_cnt[kWords + 1];
    __shared__ uint32_t s_oid[kPer * kT];
    __shared__ uint32_t s_wave[kT / 64];
    const uint32_t t = threadIdx.x;
    const uint32_t words = (cells + 1) / 2;
    for (uint32_t w = t; w < words; w += kT) s_cnt[w] = 0u;
    if (first.scene && t == 0) {
        *first.scene = S;
        first.begins[0] = 0u;
        first.begins[1] = n;
        *first.status = 0u;
    }
    __syncthreads();
    uint32_t k[kPer], rank[kPer], id[kPer];
    uint32_t flags = 0;
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const uint32_t i = t + (uint32_t)j * kT;
        k[j] = 0u;
        id[j] = i;
        if (i < n) {
            if (first.scene) {
                const float4 p = pos_a[i];
                k[j] = cell_key(S, p.x, p.y, p.z, flags);
            } else {
                k[j] = key[i];
                id[j] = oid_a[i];
            }
        }
    }
    if (flags) atomicOr(first.status, flags);   // after thread 0's store: a barrier lies between
#pragma unroll
    for (int j = 0; j < kPer; ++j)
        if (t + (uint32_t)j * kT < n) {
            const uint32_t sh = 16u * (k[j] & 1u);
            rank[j] = atomicAdd(&s_cnt[k[j] >> 1], 1u << sh) >> sh & 0xFFFFu;
        }
    __syncthreads();
    // cell starts in place of the counts; an odd number of words per thread
    // keeps the lanes on different banks
    const uint32_t per = ((words + kT - 1) / kT) | 1u;
    const uint32_t w0 = min(t * per, words), w1 = min(w0 + per, words);
    uint32_t sum = 0;
    for (uint32_t w = w0; w < w1; ++w) sum += (s_cnt[w] & 0xFFFFu) + (s_cnt[w] >> 16);
    uint32_t at = scan_block(sum, s_wave);
    for (uint32_t w = w0; w < w1; ++w) {
        const uint32_t c = s_cnt[w], lo = c & 0xFFFFu;
        s_cnt[w] = at | (at + lo) << 16;
        at += lo + (c >> 16);
    }
    __syncthreads();
    auto begin = [&](uint32_t c) { return half_of(s_cnt, c); };
    auto end = [&](uint32_t c) { return c + 1 < cells ? half_of(s_cnt, c + 1) : n; };
#pragma unroll
    for (int j = 0; j < kPer; ++j)
        if (t + (uint32_t)j * kT < n) s_oid[begin(k[j]) + rank[j]] = id[j];
    for (uint32_t c = t; c < cells; c += kT) {
        const int b = (int)begin(c), e = (int)end(c);
        range[c] = e > b ? make_int2(b, e) : make_int2(-1, -1);
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const uint32_t i = t + (uint32_t)j * kT;
        if (i < n) {
            const uint32_t b = begin(k[j]), e = end(k[j]);
            uint32_t dst = b;
            for (uint32_t q = b; q < e; ++q) dst += s_oid[q] < id[j] ? 1u : 0u;
            skey[dst] = k[j];
            pos_b[dst] = pos_a[i];
            vel_b[dst] = vel_a[i];
            oid_b[dst] = id[j];
            if (state_a) state_b[dst] = state_a[i];
            if (slot_of_oid) slot_of_oid[id[j]] = dst;
        }
    }
}

}  // namespace

bool small_sort(uint32_t n, uint64_t cells) { return n <= (uint32_t)(kPer * kT) && cells <= kMaxCells; }

void launch_small_sort(hipStream_t st, const StepBuffers& b, uint32_t cells, const DevScene& S, const SmallFirst& f) {
    hipLaunchKernelGGL(k_small_sort, dim3(1), dim3(kT), 0, st, S, f, b.key, b.oid_a, b.pos_a, b.vel_a, b.state_a, b.n,
                       cells, b.range, b.skey, b.pos_b, b.vel_b, b.oid_b, b.state_b, b.slot_of_oid);
}

}  // namespace sph
