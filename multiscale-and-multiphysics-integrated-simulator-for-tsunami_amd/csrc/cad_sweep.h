// cad_sweep.h -- what the two pipelined forms of the MILU sweeps share: buffer
// accesses, the mailbox entries tiles hand values on with, the marker of
// inactive cells.  Included by cad_sweep.hip and cad_wave_sweep.hip.
#pragma once
#include "cad_common.h"

namespace {

constexpr unsigned SPIN_LIMIT = 1u << 20;
constexpr unsigned OOB = 0xFFFFFFF0u;
constexpr int CPOL_DEVICE = 16;      // sc1: device-scope coherent access
// inactive-cell marker: a signalling-NaN pattern that no arithmetic produces
constexpr unsigned long long MARK = 0x7FF4DEADBEEF0001ull;

typedef unsigned v4u __attribute__((ext_vector_type(4)));
typedef unsigned v3u __attribute__((ext_vector_type(3)));
typedef unsigned v2u __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) void lds_void;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void *p, unsigned long long bytes)
{
    const unsigned nrec = bytes > 0xFFFFFFF0ull ? 0xFFFFFFF0u : (unsigned)bytes;
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, (int)nrec, 0x00020000);
}

// 16 bytes per lane from buffer offset off straight into LDS at lds + 16*lane
__device__ __forceinline__ void load_lds16(__amdgpu_buffer_rsrc_t r, void *lds, unsigned off)
{
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void *)lds, 16, off, 0, 0, 0);
}

__device__ __forceinline__ bool is_mark(double x)
{
    return __builtin_bit_cast(unsigned long long, x) == MARK;
}

// {value, sequence number} of a mailbox entry: 12 bytes inside the 16-byte
// entry that one store wrote
__device__ __forceinline__ v3u mb_load(__amdgpu_buffer_rsrc_t r, unsigned off)
{
    return __builtin_amdgcn_raw_buffer_load_b96(r, off, 0, CPOL_DEVICE);
}

__device__ __forceinline__ void mb_store(__amdgpu_buffer_rsrc_t r, unsigned off, double x, unsigned seq)
{
    const v2u b = __builtin_bit_cast(v2u, x);
    const v4u e = {b.x, b.y, seq, seq};
    __builtin_amdgcn_raw_buffer_store_b128(e, r, off, 0, CPOL_DEVICE);
}

// The tiles in the dependency order of the sweeps: by anti-diagonal bj + bk,
// then by bj.
__global__ void k_tile_order(int ntj, int ntk, int *order)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= ntj * ntk) return;
    const int bj = t % ntj, diag = t % ntj + t / ntj;
    int pos = 0;
    for (int s = 0; s < diag; s++) pos += min(ntj - 1, s) - max(0, s - (ntk - 1)) + 1;
    order[pos + bj - max(0, diag - (ntk - 1))] = t;
}

}  // namespace
