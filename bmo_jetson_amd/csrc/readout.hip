// readout.hip -- ring slots of one session to and from ggml's block_q4_0.
//
// A readout's blocks, [slots][n_kv_heads][head_dim / 32] of 18 bytes, lie in
// the ring as 16 code bytes here and a 2-byte scale there, 2304-byte groups
// of each kv head far apart.  One thread moves one block between the ring and
// LDS, and a workgroup's 256 blocks (4608 contiguous bytes, whole 16-byte
// pieces) move between LDS and the caller's side of a pinned host buffer
// coalesced, so the blocks cross the host link once and as large transfers.
// Bound: that link, the waits around the launch and the host's own copy out
// of the pinned buffer.  (A 512-slot, 32-head layer's K or V, 1.2 MB: 88 us a
// call; group by group with hipMemcpy and converted on the host it took 1024
// copies, 15 ms out and 25 ms in.)
#include "kernels.hpp"

namespace bmo {

namespace {

constexpr int kBlockBytes = 18;
constexpr int kWgBlocks = 256;
constexpr int kWgPieces = kWgBlocks * kBlockBytes / 16;
static_assert(kWgBlocks * kBlockBytes % 16 == 0, "whole pieces");

// Block e of the readout: its slot's code bytes and its scale's two bytes.
struct Place {
    uint4 *codes;
    uint16_t *scale;
};
__device__ __forceinline__ Place place(const ReadoutParams &p, int64_t e) {
    const int nblk = p.g.head_dim / kQK;
    const int blk = (int) (e % nblk);
    const int64_t row = e / nblk;
    const int h = (int) (row % p.g.n_kv_heads);
    const int slot = p.slot0 + (int) (row / p.g.n_kv_heads);
    uint8_t *stripe = p.base + p.g.stripe_offset(p.layer, p.session, h);
    return Place{reinterpret_cast<uint4 *>(stripe + (p.which ? p.g.vcode_offset(slot, blk) : p.g.kcode_offset(slot, blk))),
                 reinterpret_cast<uint16_t *>(stripe + p.g.scale_offset(slot, blk)) + p.which};
}

}  // namespace

__global__ __launch_bounds__(kWgBlocks) void export_kernel(ReadoutParams p) {
    __shared__ __align__(16) uint16_t s[kWgBlocks * kBlockBytes / 2];
    const int64_t e0 = (int64_t) blockIdx.x * kWgBlocks;
    const int64_t e = e0 + threadIdx.x;
    if (e < p.n_blocks) {
        const Place q = place(p, p.first + e);
        const uint32_t flip = p.which ? 0u : 0x88888888u;
        const uint4 c = *q.codes;
        const uint32_t w[4] = {c.x ^ flip, c.y ^ flip, c.z ^ flip, c.w ^ flip};
        uint16_t *d = s + threadIdx.x * (kBlockBytes / 2);
        d[0] = *q.scale;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            d[1 + 2 * i] = (uint16_t) w[i];
            d[2 + 2 * i] = (uint16_t) (w[i] >> 16);
        }
    }
    __syncthreads();
    // whole pieces: the buffer ends at a workgroup's end
    uint4 *dst = reinterpret_cast<uint4 *>(p.blocks + e0 * kBlockBytes);
    for (int i = threadIdx.x; i < kWgPieces; i += kWgBlocks) dst[i] = reinterpret_cast<const uint4 *>(s)[i];
}

__global__ __launch_bounds__(kWgBlocks) void import_kernel(ReadoutParams p) {
    __shared__ __align__(16) uint16_t s[kWgBlocks * kBlockBytes / 2];
    const int64_t e0 = (int64_t) blockIdx.x * kWgBlocks;
    const uint4 *src = reinterpret_cast<const uint4 *>(p.blocks + e0 * kBlockBytes);
    for (int i = threadIdx.x; i < kWgPieces; i += kWgBlocks) reinterpret_cast<uint4 *>(s)[i] = src[i];
    __syncthreads();
    const int64_t e = e0 + threadIdx.x;
    if (e >= p.n_blocks) return;
    const uint16_t *d = s + threadIdx.x * (kBlockBytes / 2);
    const uint32_t flip = p.which ? 0u : 0x88888888u;
    uint32_t w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = (d[1 + 2 * i] | ((uint32_t) d[2 + 2 * i] << 16)) ^ flip;
    const Place q = place(p, p.first + e);
    *q.codes = make_uint4(w[0], w[1], w[2], w[3]);
    *q.scale = d[0];
}

int64_t readout_buffer_bytes(int64_t n_blocks) {
    return (n_blocks + kWgBlocks - 1) / kWgBlocks * (kWgBlocks * kBlockBytes);
}

hipError_t launch_readout(const ReadoutParams &p, bool to_ring, hipStream_t stream) {
    const unsigned wgs = (unsigned) ((p.n_blocks + kWgBlocks - 1) / kWgBlocks);
    ReadoutParams arg = p;
    void *args[] = {&arg};
    const void *kernel = to_ring ? reinterpret_cast<const void *>(import_kernel) : reinterpret_cast<const void *>(export_kernel);
    return hipLaunchKernel(kernel, dim3(wgs), dim3(kWgBlocks), args, 0, stream);
}

}  // namespace bmo
