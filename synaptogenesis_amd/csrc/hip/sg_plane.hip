// Base activator for spiking (BIT) sources with finite weights, driven by a
// spike plane.
//
// For a BIT source the reference's per-synapse value is
// extract(word, delay) * w = (0 or 1) * w (synapse_kernel.h:887-912,
// extractor.cpp:8-14).  With finite weights a silent synapse adds +0 or -0,
// which leaves the destination's running sum unchanged (it starts at +0 and
// a round-to-nearest sum of nonzero terms is never -0), so the sum over the
// spiking visits alone, in visit order, is the reference's sum bit for bit.
//
// 1. pack_plane_kernel turns the source's history words into a plane: the
//    bit each source neuron shows this connection (word delay/32, bit
//    31 - delay%32), 64 neurons per uint64, one wavefront ballot each.
// 2. plane_base_kernel: a block stages the plane in LDS.  Its wavefronts
//    split the visit list: each lane tests its visits' bits in LDS and
//    issues the weight loads of the spiking ones together (coalesced across
//    the tile), writing the weight -- or +0 for a silent or skipped visit --
//    to an LDS chunk.  After a barrier wavefront 0 adds the chunk in visit
//    order.  Adding +0 leaves the sum unchanged, so the result is the
//    reference's sum bit for bit.
//
// Work per synapse is a bit test in LDS; weights are read only for the
// spiking visits.  Planes larger than kPlaneMax words are read from global
// memory (through the caches) instead of LDS.
#include <hip/hip_runtime.h>

#include "sg_device.h"

namespace sg {

constexpr int kPlaneMax = 4096;     // uint64 plane words staged in LDS

typedef float f32x4 __attribute__((ext_vector_type(4)));

__global__ __launch_bounds__(256) void pack_plane_kernel(
        const uint32_t *words, int n, int delay, uint64_t *plane) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    const bool bit = i < n && ((words[i] << (delay & 31)) >> 31) != 0;
    const uint64_t m = __ballot(bit);
    // lane 0 of each wavefront: i is a multiple of 64
    if ((threadIdx.x & 63) == 0 && i < n) plane[i >> 6] = m;
}

template <int TYPE>
__device__ __forceinline__ int plane_visits(const sg_conn &c) {
    return cursor<TYPE>(c, 0).count;
}

// D destinations a block (16 or 64, inside one tile): the chain of one
// destination's additions bounds the launch, so it is kept off everything
// else as in tile_base_kernel -- a chunk's weights are on their way while
// wavefront 0 adds the chunk before, four visits to an LDS read.  Measured
// with 5 % of the sources spiking: 15 x 15 stride 2 from 256 x 320 10.8 us
// (13.0 before), from 32 x 40 7.1 us (9.6); 5000 -> 1000 fully connected 33
// us (94).
template <int TYPE, int D, int W, bool STAGED>
__global__ __launch_bounds__(64 * W) void plane_base_kernel(
        sg_conn c, const uint64_t *plane) {
    constexpr int V = 64 / D;            // visits of a wavefront load
    constexpr int PER = 8;
    constexpr int CHUNK = W * PER * V;
    constexpr int AHEAD = 4;
    static_assert(CHUNK % (4 * AHEAD) == 0, "whole reads");
    extern __shared__ uint32_t splane[];          // STAGED: the plane
    __shared__ f32x4 vals[2][CHUNK / 4][D];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int d = lane % D, kk = lane / D;
    const int slot = blockIdx.x * D + d;
    const bool live = slot < c.num_dest;
    const int count = plane_visits<TYPE>(c);
    const uint32_t *words = reinterpret_cast<const uint32_t *>(plane);
    if (STAGED) {
        const int np = (c.from_size + 31) >> 5;
        for (int i = threadIdx.x; i < np; i += 64 * W) splane[i] = words[i];
        __syncthreads();
        words = splane;
    }
    const float *wbase = c.convolutional
        ? c.weights
        : c.weights + tiled_index(live ? slot : 0, 0, c.k_per_dest);
    const long wstep = c.convolutional ? 1 : 64;
    const int first = wave * PER * V + kk;
    SynapseIter<TYPE> start;
    start.init(c, live ? slot : 0);
    float v[PER];
    auto issue = [&](int k0) {
        SynapseIter<TYPE> it = start;
        it.jump(k0 + first);
        uint32_t on = 0;
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const int k = k0 + first + j * V;
            const int from = live && k < count ? it.source() : -1;
            if (from >= 0)
                on |= ((words[from >> 5] >> (from & 31)) & 1u) << j;
#pragma unroll
            for (int b = 0; b < V; ++b) it.advance();
        }
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            v[j] = 0.0f;
            if ((on >> j) & 1u) v[j] = wbase[(k0 + first + j * V) * wstep];
        }
    };
    auto store = [&](int buf) {
        if (V == 1) {
#pragma unroll
            for (int j = 0; j < PER; j += 4) {
                const f32x4 q = {v[j], v[j + 1], v[j + 2], v[j + 3]};
                vals[buf][(wave * PER + j) / 4][d] = q;
            }
        } else {
            float *q = reinterpret_cast<float *>(vals[buf]);
#pragma unroll
            for (int j = 0; j < PER; ++j) {
                const int at = first + j * V;
                q[((at >> 2) * D + d) * 4 + (at & 3)] = v[j];
            }
        }
    };
    float sum = 0.0f;
    if (count > 0) {
        issue(0);
        store(0);
    }
    for (int k0 = 0, buf = 0; k0 < count; k0 += CHUNK, buf ^= 1) {
        __syncthreads();
        const bool more = k0 + CHUNK < count;
        if (more) issue(k0 + CHUNK);
        if (wave == 0) {
            // entries past the count hold +0
            const int groups = (min(CHUNK, count - k0) + 3) / 4;
            for (int g = 0; g < groups; g += AHEAD) {
                f32x4 q[AHEAD];
#pragma unroll
                for (int i = 0; i < AHEAD; ++i) q[i] = vals[buf][g + i][d];
#pragma unroll
                for (int i = 0; i < AHEAD; ++i) {
                    sum += q[i][0];
                    sum += q[i][1];
                    sum += q[i][2];
                    sum += q[i][3];
                }
            }
        }
        if (more) store(buf ^ 1);
    }
    if (live && wave == 0 && kk == 0)
        put_sum(c, slot_to_index(c, slot), sum);
}

// Fully connected, at most kListMax sources: every destination visits the
// sources in index order, so the spiking ones form one list shared by the
// whole layer.  A block (one wavefront, one tile of 64 destinations)
// builds it in LDS from the plane -- a popcount per plane word, a
// wavefront prefix sum over the words, each word's set bits written at its
// offset -- and then each lane adds its weights of the listed sources in
// list order (the same 256-byte row of the tiled weights for all lanes per
// entry).  Silent visits add +0 in the reference's loop, so the sum is its
// sum bit for bit.
constexpr int kListMax = 4096;

__global__ __launch_bounds__(64) void fc_list_kernel(sg_conn c,
                                                     const uint64_t *plane) {
    __shared__ int list[kListMax];
    __shared__ int total;
    const int lane = threadIdx.x;
    const int np = (c.from_size + 63) >> 6;          // <= 64 words
    const uint64_t word = lane < np ? plane[lane] : 0ull;
    const int n = __popcll(word);
    int pre = n;                                      // inclusive scan
    for (int d = 1; d < 64; d <<= 1) {
        const int v = __shfl_up(pre, d, 64);
        if (lane >= d) pre += v;
    }
    int at = pre - n;
    for (uint64_t m = word; m; m &= m - 1)
        list[at++] = lane * 64 + (int)__builtin_ctzll(m);
    if (lane == 63) total = pre;
    __syncthreads();
    const int m = total;
    const int slot = blockIdx.x * 64 + lane;
    if (slot >= c.num_dest) return;
    const float *wrow = c.weights + tiled_index(slot, 0, c.k_per_dest);
    float sum = 0.0f;
    int j = 0;
    for (; j + 8 <= m; j += 8) {
        float v[8];
#pragma unroll
        for (int b = 0; b < 8; ++b) v[b] = wrow[(long)list[j + b] * 64];
#pragma unroll
        for (int b = 0; b < 8; ++b) sum += v[b];
    }
    for (; j < m; ++j) sum += wrow[(long)list[j] * 64];
    put_sum(c, slot_to_index(c, slot), sum);
}

template <int TYPE, int D, int W>
static hipError_t launch_plane_w(const sg_conn &c, hipStream_t st) {
    dim3 g((c.num_dest + D - 1) / D), b(64 * W);
    const int np = (c.from_size + 63) / 64;
    if (np <= kPlaneMax)
        hipLaunchKernelGGL((plane_base_kernel<TYPE, D, W, true>), g, b,
                           (size_t)np * 8, st, c, c.plane);
    else
        hipLaunchKernelGGL((plane_base_kernel<TYPE, D, W, false>), g, b, 0,
                           st, c, c.plane);
    return hipGetLastError();
}

// One lane per destination: it walks its visits in order, sixteen at a
// time, reading the plane words through the caches (no LDS staging, no
// barrier: a block is one short wavefront).  Every visit's plane word is
// loaded first, then the weights of the spiking visits, then the sum in
// visit order (silent visits add +0).
template <int TYPE>
__global__ __launch_bounds__(64) void plane_lane_kernel(sg_conn c,
                                                        const uint64_t *plane) {
    constexpr int V = 16;
    const int slot = blockIdx.x * 64 + threadIdx.x;
    if (slot >= c.num_dest) return;
    const int count = plane_visits<TYPE>(c);
    const float *wbase = c.convolutional
        ? c.weights : c.weights + tiled_index(slot, 0, c.k_per_dest);
    const long wstep = c.convolutional ? 1 : 64;
    const uint32_t *words = reinterpret_cast<const uint32_t *>(plane);
    SynapseIter<TYPE> it;
    it.init(c, slot);
    float sum = 0.0f;
    for (int k0 = 0; k0 < count; k0 += V) {
        int from[V];
        uint32_t word[V];
#pragma unroll
        for (int b = 0; b < V; ++b) {
            from[b] = -1;
            if (k0 + b < count) {
                from[b] = it.source();
                it.advance();
            }
            word[b] = from[b] >= 0 ? words[from[b] >> 5] : 0u;
        }
        float v[V];
#pragma unroll
        for (int b = 0; b < V; ++b) {
            v[b] = 0.0f;
            if ((word[b] >> (from[b] & 31)) & 1u)
                v[b] = wbase[(k0 + b) * wstep];
        }
#pragma unroll
        for (int b = 0; b < V; ++b) sum += v[b];
    }
    put_sum(c, slot_to_index(c, slot), sum);
}

// A lane per destination for up to 16 visits, and for more once the layer's
// own wavefronts fill the GPU, the later the more visits there are: 25 visits
// at 1024 tiles 9.3 us against 9.6 with eight wavefronts a tile, 49 at 1407
// 14.8 against 13.8 and at 2025 15.9 against 18.3, 81 at 2500 28 against 26 and
// at 2757 29 against 44.  SPARSE, whose indices a lane waits for: 30 visits at
// 1563 tiles 11.5 against 10.2 and at 3125 18.5 against 22.8, 64 at 3125 30
// against 25 and at 7813 48 against 49.
static bool plane_lanes(int type, int count, int tiles) {
    if (count <= 16) return true;
    if (type == SG_SPARSE)
        return count <= 64 && tiles >= (count <= 32 ? 2048 : 4096);
    if (count <= 64) return tiles >= 1024 + 16 * (count > 25 ? count - 25 : 0);
    return count <= 128 && tiles >= 2560;
}

// Which form (all give the same bits), by one sweep:
// * a lane per destination (plane_lanes);
// * 16 destinations a block while that gives every block a CU of its own
//   (64 tiles) and its chunk has more visits than one of sixteen wavefronts a
//   tile: 21 x 21 on 64 x 64 11 us against 14, 11 x 11 9.3 against 7.8;
// * beside a long kernel on another stream (sg_conn.beside), four
//   wavefronts a tile: they start as soon as a CU has four free wave slots;
// * sixteen wavefronts a tile up to two tiles a CU (15 x 15 on 128 x 128
//   7.7 us against 10 with eight), eight beyond (on 256 x 256 17.9 against
//   19.5), four of those blocks a CU; SPARSE also sixteen where a few tiles
//   are left to a last round of eight (1032 tiles: 250 visits 34 us against 39,
//   600 visits 85 against 105; 1563 tiles 45 against 41).
template <int TYPE>
static hipError_t launch_plane_t(const sg_conn &c, hipStream_t st) {
    const int count = cursor<TYPE>(c, 0).count;
    const int tiles = (c.num_dest + 63) / 64;
    if (plane_lanes(TYPE, count, tiles)) {
        hipLaunchKernelGGL(plane_lane_kernel<TYPE>, dim3(tiles), dim3(64), 0,
                           st, c, c.plane);
        return hipGetLastError();
    }
    if (count > 128 && tiles <= 64) return launch_plane_w<TYPE, 16, 16>(c, st);
    if (c.beside) return launch_plane_w<TYPE, 64, 4>(c, st);
    const bool few_left = TYPE == SG_SPARSE && count > 64 && tiles > 1024 &&
                          tiles < 3072 && (tiles - 1) % 1024 < 256;
    if (tiles <= 512 || few_left) return launch_plane_w<TYPE, 64, 16>(c, st);
    return launch_plane_w<TYPE, 64, 8>(c, st);
}

// True when the plane path applies: a BIT source, finite weights and a
// tiled connection type.
bool plane_path(const sg_conn &c) {
    return c.plane != nullptr && c.skip_silent && c.out_type == SG_OUT_BIT &&
           c.type != SG_ONE_TO_ONE;
}

hipError_t launch_plane_base(const sg_conn &c, hipStream_t st) {
    if (!c.plane_ready) {
        const int n = c.from_size;
        hipLaunchKernelGGL(pack_plane_kernel, dim3((n + 255) / 256),
                           dim3(256), 0, st, c.src, n, c.delay, c.plane);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    switch (c.type) {
        case SG_FULLY_CONNECTED:
            if (c.from_size <= kListMax && !c.convolutional) {
                hipLaunchKernelGGL(fc_list_kernel, dim3((c.num_dest + 63) / 64),
                                   dim3(64), 0, st, c, c.plane);
                return hipGetLastError();
            }
            return launch_plane_t<SG_FULLY_CONNECTED>(c, st);
        case SG_SUBSET: return launch_plane_t<SG_SUBSET>(c, st);
        case SG_CONVERGENT: return launch_plane_t<SG_CONVERGENT>(c, st);
        case SG_DIVERGENT: return launch_plane_t<SG_DIVERGENT>(c, st);
        case SG_SPARSE: return launch_plane_t<SG_SPARSE>(c, st);
    }
    return hipErrorInvalidValue;
}

}  // namespace sg

using namespace sg;

extern "C" int sg_hip_pack_plane(const uint32_t *words, int n, int delay,
                                 uint64_t *plane, void *stream) {
    if (n <= 0) return 0;
    hipLaunchKernelGGL(pack_plane_kernel, dim3((n + 255) / 256), dim3(256), 0,
                       (hipStream_t)stream, words, n, delay, plane);
    return hipGetLastError();
}
