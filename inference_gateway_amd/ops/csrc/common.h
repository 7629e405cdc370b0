// Common helpers for MI355X (gfx950 / CDNA4) HIP kernels.
//
// Design notes: CDNA4 wavefront is 64 lanes; block dims are multiples of 64.
// All kernels here are written directly for gfx950 — no CUDA compatibility
// paths, no Triton. bf16 is the primary activation dtype.
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>
#include <stdint.h>

#define WAVE_SIZE 64

#define DEVINLINE __device__ __forceinline__

// ---------------------------------------------------------------------------
// bf16 <-> f32
// ---------------------------------------------------------------------------
DEVINLINE float bf16_to_f32(uint16_t h) {
  union {
    uint32_t u;
    float f;
  } v;
  v.u = ((uint32_t)h) << 16;
  return v.f;
}

DEVINLINE uint16_t f32_to_bf16(float f) {
  union {
    float f;
    uint32_t u;
  } v;
  v.f = f;
  // round-to-nearest-even
  uint32_t lsb = (v.u >> 16) & 1;
  v.u += 0x7fffu + lsb;
  return (uint16_t)(v.u >> 16);
}

// packed vector types for wide loads
typedef uint32_t u32;
typedef uint16_t u16;
struct alignas(16) ushort8 {
  uint16_t v[8];
};
struct alignas(8) ushort4x {
  uint16_t v[4];
};

// ---------------------------------------------------------------------------
// Wave-level reductions (64-wide).
// ---------------------------------------------------------------------------
DEVINLINE float wave_reduce_sum(float x) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    x += __shfl_xor(x, off, WAVE_SIZE);
  }
  return x;
}

DEVINLINE float wave_reduce_max(float x) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    x = fmaxf(x, __shfl_xor(x, off, WAVE_SIZE));
  }
  return x;
}

// Reduce over a contiguous group of `width` lanes (width must be power of 2).
template <int WIDTH>
DEVINLINE float group_reduce_sum(float x) {
#pragma unroll
  for (int off = WIDTH / 2; off > 0; off >>= 1) {
    x += __shfl_xor(x, off, WAVE_SIZE);
  }
  return x;
}

template <int WIDTH>
DEVINLINE float group_reduce_max(float x) {
#pragma unroll
  for (int off = WIDTH / 2; off > 0; off >>= 1) {
    x = fmaxf(x, __shfl_xor(x, off, WAVE_SIZE));
  }
  return x;
}

// Block-level reduce using LDS scratch; BLOCK must be multiple of 64.
// `lds` must have at least BLOCK/64 floats. Result valid on all threads.
template <int BLOCK>
DEVINLINE float block_reduce_sum(float x, float* lds) {
  const int nwaves = BLOCK / WAVE_SIZE;
  int lane = threadIdx.x & (WAVE_SIZE - 1);
  int wave = threadIdx.x >> 6;
  x = wave_reduce_sum(x);
  if (lane == 0) lds[wave] = x;
  __syncthreads();
  float r = (threadIdx.x < nwaves) ? lds[threadIdx.x] : 0.0f;
#pragma unroll
  for (int off = 1; off < nwaves; off <<= 1) {
    r += __shfl_xor(r, off, WAVE_SIZE);
  }
  // broadcast from lane 0 of wave 0 via lds
  if (threadIdx.x == 0) lds[0] = r;
  __syncthreads();
  return lds[0];
}

// A rotated pair (x1, x2) of NeoX RoPE, rounded.  Written out, so that every kernel
// has the same bits.
DEVINLINE void rope_pair(uint16_t& x1, uint16_t& x2, float cos, float sin) {
  const float a = bf16_to_f32(x1), b = bf16_to_f32(x2);
  x1 = f32_to_bf16(fmaf(a, cos, -(b * sin)));
  x2 = f32_to_bf16(fmaf(b, cos, a * sin));
}

// The gate of a gated activation, act(g): GATE 1 SiLU, 2 GELU by its tanh form
// (0: the product has no activation), (1 + tanh(x)) / 2 being sigmoid(2 x).
template <int GATE>
DEVINLINE float gate_act(float g) {
  if constexpr (GATE == 2)
    return g / (1.0f + __expf(-1.5957691216057308f *
                              (g + 0.044715f * g * g * g)));
  else
    return g / (1.0f + __expf(-g));
}

// Lines of memory to operands of the 16x16x32 matrix instructions.
//
// A load takes whole 128-byte lines, eight lanes a line; a matrix operand wants
// neighbouring lanes in neighbouring rows.  The 16 lines of two loads (rows 0-7
// and 8-15, 64 bf16 of each) go through 2 KB of LDS of the wave's own and come
// back as the operands of their first and second 32 entries.  The 16-byte pieces
// of a row are permuted by it, so that neither access meets itself in a bank.
// The wave's other lanes write what a lane reads: the fences keep the compiler
// from moving an access past another, the LDS keeps a wave's order by itself.
struct LineTurn {
  typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
  int put, put_hi, get, get_hi;
  static DEVINLINE int perm(int row) { return (row & 3) | ((row >> 3) & 1) << 2; }
  DEVINLINE explicit LineTurn(int lane) {
    const int r8 = lane >> 3, r16 = lane & 15, quad = lane >> 4;
    put = r8 * 8 + ((lane & 7) ^ perm(r8));
    put_hi = 64 + r8 * 8 + ((lane & 7) ^ perm(8 + r8));
    get = r16 * 8 + (quad ^ perm(r16));
    get_hi = r16 * 8 + ((4 + quad) ^ perm(r16));
  }
  static DEVINLINE void fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
  DEVINLINE void operator()(u32x4* t, const u32x4& in0, const u32x4& in1,
                            u32x4& out0, u32x4& out1) const {
    fence();
    t[put] = in0;
    t[put_hi] = in1;
    fence();
    out0 = t[get];
    out1 = t[get_hi];
  }
};

#define HIP_CHECK_KERNEL()                                                     \
  do {                                                                         \
    hipError_t err = hipGetLastError();                                        \
    if (err != hipSuccess) {                                                   \
      TORCH_CHECK(false, "HIP kernel launch failed: ", hipGetErrorString(err)); \
    }                                                                          \
  } while (0)
