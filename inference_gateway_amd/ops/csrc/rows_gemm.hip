// y = x W^T for the tens of rows of x of a decode step or a short prompt,
// gfx950, bf16, products and sums in fp32 (16x16x32 matrix instructions).
//
// Bound by streaming W once from HBM.  A wave owns 16 rows of W and takes them
// from memory straight to registers, 512 bytes of each per slice of K, two
// slices on their way while one is multiplied; the slice's rows of x go
// through LDS once for the eight waves of a workgroup.
//
// Eight neighbouring lanes load a whole 128-byte line.  A matrix operand wants
// neighbouring lanes in neighbouring rows, but a load laid out like that is 64
// requests of 16 bytes to the compute unit's cache, which takes 65 cycles for
// it: 28 KB a microsecond for a compute unit, even from L2.  In whole lines it is
// 92, so the lines go through 2 KB of LDS of the wave's own to be turned.
//
// Workgroups start at different slices, waves at different lines: rows of W lie
// a multiple of 4 KB apart and would meet in the same memory channels (28672 x
// 4096, 16 rows, before the lines were turned: 52.0 us, with the starts apart
// 48.0).
//
// W is read once a step, and in rows of 4 KB and more by nontemporal loads (RG_ONCE):
// others leave it in the memory side's cache, which has no room for a model, and that
// costs the memory a ninth of its rate (loads alone, 128256 rows of 8 KB in this pattern,
// 183 and 157 us, 28672 of them 45.0 and 39.4; a row at a time, 1 KB a load, 168 and 150).
// Shorter rows are slower so (28672 x 1024 as SwiGLU, 9 / 17 / 33 rows, plain and so, 12.9
// 13.4 13.8 and 13.9 14.0 14.2).  Of 49 rows and more the kernel waits for other things,
// and between the others of a step plain loads are as good (28672 x 4096 as SwiGLU 47.0
// and 47.3 us, 43 rows 44.3 and 42.3; 128256 x 4096, 61 rows, 194 and 199).
//
// GATE: a wave's 16 rows are eight gate rows and the up rows of the same outputs,
// and the result is act(gate) * up of the fp32 sums.
//
// Measured, here and with operands loaded as the matrix unit wants them (us, W
// cold; 16 / 32 / 43 / 64 rows): 28672 x 4096 as SwiGLU 42.2 43.0 43.8 45.7 (5.1
// TB/s) and 45.7 46.9 48.6 51.0; 28672 x 4096 at 32 / 43 / 64 rows 42.7 44.8 45.8
// and 48.0 50.7 51.0; 128256 x 4096 178 182 189 (5.6 TB/s) and 188 193 201; 4096 x
// 14336 27.7 29.5 32.7 and 29.9 31.2 34.1.  The library, 32 / 48 / 64 rows: 56 64
// 55, 200 210 213 and 34 40 41.  These are one after the other on one card; on
// another 45.3 46.0 46.3 48.8 as SwiGLU and 186 191 195 for 128256 x 4096.  narrow_gemm,
// asked first, takes more than 48 rows of the former and the latter.
#include <ATen/cuda/CUDAContext.h>
#include <c10/cuda/CUDAGuard.h>
#include <torch/extension.h>

#include <type_traits>

#include "common.h"

namespace igw {

typedef __attribute__((ext_vector_type(8))) __bf16 rg_bf16x8;
typedef __attribute__((ext_vector_type(4))) float rg_f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t rg_u32x4;

constexpr int RG_BK = 256;     // entries of a K slice
constexpr int64_t RG_ONCE = 2048;   // entries of a row of W, nontemporal from there on
constexpr int RG_WAVES = 8;

struct RowsArgs {
  uint16_t* out;         // [M, N]
  float* part;           // [S, M, N] sums of a split K, or null
  const uint16_t* x;
  const uint16_t* w;
  const uint16_t* bias;
  int M, N, K;
  int64_t x_rs;
};

template <int MT, int GATE, bool ONCE>
__global__ __launch_bounds__(64 * RG_WAVES, 2) void rows_gemm_kernel(
    RowsArgs a) {
  __shared__ __attribute__((aligned(1024))) uint16_t xs[3][MT * 16 * RG_BK];
  __shared__ __attribute__((aligned(1024))) rg_u32x4 turned[RG_WAVES][2][128];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, quad = lane >> 4;
  const int slices = a.K / RG_BK;
  const int s0 = slices * blockIdx.y / gridDim.y;
  const int last = slices * (blockIdx.y + 1) / gridDim.y - 1;
  const int rot = (blockIdx.x + (blockIdx.x >> 3)) % (last + 1 - s0);
  constexpr bool SWIGLU = GATE != 0;
  constexpr int COLS = SWIGLU ? 8 : 16;    // outputs of a wave
  const int n0 = (blockIdx.x * RG_WAVES + wave) * COLS;

  // Matrix row r of a wave's tile is this row of W; with a gate four of them
  // are two gate rows and the up rows of the same two outputs.
  auto w_row = [&](int r) {
    return a.w + (int64_t)(SWIGLU ? min(n0 + (r >> 2) * 2 + (r & 1), a.N - 1) +
                                        ((r >> 1) & 1) * a.N
                                  : min(n0 + r, a.N - 1)) *
                     a.K;
  };
  // A load takes whole 128-byte lines: eight rows, eight lanes a row.
  const int piece = (lane & 7) * 8;
  const uint16_t* w_lo = w_row(lane >> 3) + piece;
  const uint16_t* w_hi = w_row(8 + (lane >> 3)) + piece;
  const LineTurn turn_lines(lane);
  // rows of x: 512 bytes of a row per 32 lanes, its 16-byte pieces permuted by
  // the row so that the 16 rows of a matrix operand lie in different banks
  constexpr int XR = MT * 8 / RG_WAVES;    // 16-byte pieces of x per lane
  const uint16_t* xp[XR];
#pragma unroll
  for (int i = 0; i < XR; ++i) {
    const int row = (i * RG_WAVES + wave) * 2 + (lane >> 5);
    xp[i] = a.x + min(row, a.M - 1) * a.x_rs + (lane & 31) * 8;
  }
  // a slice of x and of W, x first as it is waited for first; past the end the
  // last slice once more, so that the loop is the same to its end
  auto load = [&](rg_u32x4 (&xr)[XR], rg_u32x4 (&wr)[8], int sl) {
    int at = min(sl, last) + rot;
    at = at > last ? at - (last + 1 - s0) : at;
    const int k = at * RG_BK;
#pragma unroll
    for (int i = 0; i < XR; ++i)
      xr[i] = *reinterpret_cast<const rg_u32x4*>(xp[i] + k);
    asm volatile("" ::: "memory");
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const auto* p = reinterpret_cast<const rg_u32x4*>(
          (j & 1 ? w_hi : w_lo) + k + ((j / 2 + wave) & 3) * 64);
      wr[j] = ONCE ? __builtin_nontemporal_load(p) : *p;
    }
    asm volatile("" ::: "memory");
  };
  auto put_x = [&](const rg_u32x4 (&xr)[XR], uint16_t* s) {
#pragma unroll
    for (int i = 0; i < XR; ++i) {
      const int row = (i * RG_WAVES + wave) * 2 + (lane >> 5);
      *reinterpret_cast<rg_u32x4*>(
          s + row * RG_BK + ((lane & 31) ^ (row & 15)) * 8) = xr[i];
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  rg_f32x4 acc[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) acc[m] = rg_f32x4{0.f, 0.f, 0.f, 0.f};
  // Lines are turned one step ahead of their products, in two buffers in turn;
  // a wave's LDS accesses keep their order.
  auto compute = [&](const rg_u32x4 (&wr)[8], const uint16_t* s) {
    rg_u32x4 half[2][2];
    auto turn = [&](int j) __attribute__((always_inline)) {
      turn_lines(turned[wave][j & 1], wr[2 * j], wr[2 * j + 1], half[j & 1][0],
                 half[j & 1][1]);
    };
    turn(0);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (j < 3) turn(j + 1);
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          const int chunk = (((j + wave) & 3) * 8 + h * 4 + quad) ^ r16;
          const rg_bf16x8 xv = *reinterpret_cast<const rg_bf16x8*>(
              s + (m * 16 + r16) * RG_BK + chunk * 8);
          acc[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(rg_bf16x8, half[j & 1][h]), xv, acc[m], 0, 0,
              0);
        }
    }
  };

  // Past the barrier of put_x a slice's rows of x are there for every wave; the
  // buffer that they go to was last read two barriers before.
  rg_u32x4 x0[XR], x1[XR], x2[XR], w0[8], w1[8], w2[8];
  load(x0, w0, s0);
  load(x1, w1, s0 + 1);
  put_x(x0, xs[0]);
  for (int sl = s0;; sl += 3) {
    load(x2, w2, sl + 2);
    compute(w0, xs[0]);
    if (sl >= last) break;
    put_x(x1, xs[1]);
    load(x0, w0, sl + 3);
    compute(w1, xs[1]);
    if (sl + 1 >= last) break;
    put_x(x2, xs[2]);
    load(x1, w1, sl + 4);
    compute(w2, xs[2]);
    if (sl + 2 >= last) break;
    put_x(x0, xs[0]);
  }

#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const int row = m * 16 + r16;
    if (row >= a.M) continue;
    const rg_f32x4 y = acc[m];
    if (SWIGLU) {
      const int n = n0 + quad * 2;
      if (n >= a.N) continue;
      const uint32_t lo = f32_to_bf16(gate_act<GATE>(y[0]) * y[2]);
      const uint32_t hi = f32_to_bf16(gate_act<GATE>(y[1]) * y[3]);
      *reinterpret_cast<uint32_t*>(a.out + (int64_t)row * a.N + n) =
          lo | hi << 16;
    } else {
      const int n = n0 + quad * 4;
      if (n >= a.N) continue;
      if (a.part) {
        *reinterpret_cast<rg_f32x4*>(
            a.part + ((int64_t)blockIdx.y * a.M + row) * a.N + n) = y;
      } else {
        ushort4x o;
#pragma unroll
        for (int e = 0; e < 4; ++e)
          o.v[e] = f32_to_bf16(
              y[e] + (a.bias ? bf16_to_f32(a.bias[n + e]) : 0.0f));
        *reinterpret_cast<ushort4x*>(a.out + (int64_t)row * a.N + n) = o;
      }
    }
  }
}

// sum of the parts of a split K, with the bias
__global__ __launch_bounds__(256) void sum_parts_kernel(
    uint16_t* __restrict__ out, const float* __restrict__ part,
    const uint16_t* __restrict__ bias, int M, int N, int S) {
  const int64_t step = (int64_t)M * N;
  const int64_t at = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (at >= step) return;
  rg_f32x4 y = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
  for (int s = 0; s < S; ++s)
    y += *reinterpret_cast<const rg_f32x4*>(part + s * step + at);
  const int n = bias ? (int)(at % N) : 0;
  ushort4x o;
#pragma unroll
  for (int e = 0; e < 4; ++e)
    o.v[e] = f32_to_bf16(y[e] + (bias ? bf16_to_f32(bias[n + e]) : 0.0f));
  *reinterpret_cast<ushort4x*>(out + at) = o;
}

// out [M, N] = part [S, M, N] summed over S, plus the bias; N in fours
void sum_parts(torch::Tensor out, const torch::Tensor& part,
               const c10::optional<torch::Tensor>& bias) {
  TORCH_CHECK(part.is_cuda() && part.dim() == 3 && part.is_contiguous() &&
              part.dtype() == torch::kFloat32);
  const int64_t S = part.size(0), M = part.size(1), N = part.size(2);
  TORCH_CHECK(S < (1LL << 31) && M < (1LL << 31) && N < (1LL << 31) &&
              N % 4 == 0 && (M * N / 4 + 255) / 256 < (1LL << 31));
  TORCH_CHECK(out.dim() == 2 && out.size(0) == M && out.size(1) == N &&
              out.is_contiguous() && out.dtype() == torch::kBFloat16 &&
              (reinterpret_cast<uintptr_t>(out.data_ptr()) & 7) == 0 &&
              (reinterpret_cast<uintptr_t>(part.data_ptr()) & 15) == 0);
  TORCH_CHECK(out.device() == part.device() &&
                  (!bias.has_value() || bias->device() == part.device()),
              "tensors on different devices");
  if (bias.has_value())
    TORCH_CHECK(bias->dtype() == torch::kBFloat16 && bias->dim() == 1 &&
                bias->size(0) == N && bias->is_contiguous());
  if (M * N == 0) return;
  const at::cuda::CUDAGuard guard(part.device());
  hipLaunchKernelGGL(sum_parts_kernel, dim3((M * N / 4 + 255) / 256), dim3(256),
                     0, at::cuda::getCurrentCUDAStream(),
                     (uint16_t*)out.data_ptr(), part.data_ptr<float>(),
                     bias.has_value() ? (const uint16_t*)bias->data_ptr()
                                      : nullptr,
                     (int)M, (int)N, (int)S);
  HIP_CHECK_KERNEL();
}

// The same product where the kernel above does not fill the chip: x stays in
// registers.
//
// W is walked 16 rows at a time by a workgroup, an eighth of K (or of the
// split's part of it) by each of its eight waves, up to 512 entries, whose 16 or
// 32 rows of x lie in the wave's registers as operands from start to end.  So a
// unit of work is 128 KB of W, often in one piece, instead of 1 MB; nothing
// but the waves' sums goes through LDS, once a unit, and a wave refills the
// registers of a line of W for the next unit when it has turned it.  More than
// 32 rows are two halves, in workgroups of the same XCD at the same time (the second
// finds W in L2), or ring_gemm's below.
//
// Bound by W's bytes, and by the start for small ones (x to registers, 256 KB a
// workgroup, and the first lines: about 4 us).  Measured, library and here (us, W
// cold, 8 / 16 / 32 / 40 / 64 rows): 4096 x 4096 15.6 15.8 13.3 13.7 15.1 and 8.8
// 9.3 10.7 11.4 12.2; 6144 x 4096 14.6 14.4 15.5 17.3 18.0 and 11.3 12.0 13.7 14.0
// 15.3; 1024 x 4096 12.8 12.9 10.7 13.2 13.9 and 5.4 5.7 7.4 7.2 7.4; 4096 x 14336,
// 16 / 32 / 43 / 64 rows, the kernel above 26.1 27.7 29.5 32.7 and 24.5 25.9 29.3
// 30.8.  x loaded in the operands' layout instead of whole lines (a note above):
// 4 us more.
//
// ONCE: W is loaded past the caches of the memory's side (see above).  Not where a
// second half wants it again, and not the few MB that may have stayed there since
// the last step (HELD_ONCE: 1024 x 4096, 16 rows, 16 of them in turn, 5.7 us and
// 6.6 so; 2560 x 5120 11.9 and 11.0, 4096 x 14336 27.0 and 24.8).
constexpr int64_t HELD_ONCE = 12 << 20;   // entries of W

template <int P, int MT, int halves, bool ONCE>
__global__ __launch_bounds__(64 * RG_WAVES, 2) void held_gemm_kernel(
    RowsArgs a, int S) {
  __shared__ __attribute__((aligned(16)))
  rg_f32x4 sums[2][RG_WAVES][MT][WAVE_SIZE];
  __shared__ __attribute__((aligned(1024))) rg_u32x4 turned[RG_WAVES][2][128];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, quad = lane >> 4;
  // workgroups i and i + 8 are on the same XCD: the two halves of x
  const int half = halves == 2 ? (blockIdx.x >> 3) & 1 : 0;
  const int id = halves == 2 ? (blockIdx.x & 7) | (blockIdx.x >> 4) << 3
                             : blockIdx.x;
  const int split = id % S, step = gridDim.x / (S * halves);
  const int units = (a.N + 15) >> 4;
  int unit = id / S;
  if (unit >= step || unit >= units) return;

  // the wave's P lines of 64 entries, from another one on in each workgroup
  const int k0 = (split * RG_WAVES + wave) * P * 64;
  const int rot = ((id >> 3) + wave) % P;
  auto line = [&](int j) __attribute__((always_inline)) {
    return k0 + (j + rot >= P ? j + rot - P : j + rot) * 64;
  };
  const int r8 = lane >> 3, piece = (lane & 7) * 8;
  rg_u32x4 xf[P][2][MT], w[P][2];
#pragma unroll
  for (int j = 0; j < P; ++j)
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int m = 0; m < MT; ++m)
        xf[j][h][m] = *reinterpret_cast<const rg_u32x4*>(
            a.x + min((half * MT + m) * 16 + h * 8 + r8, a.M - 1) * a.x_rs +
            line(j) + piece);
  asm volatile("" ::: "memory");
  const uint16_t *lo, *hi;
  auto rows_of = [&](int u) __attribute__((always_inline)) {
    lo = a.w + (int64_t)min(u * 16 + r8, a.N - 1) * a.K + piece;
    hi = a.w + (int64_t)min(u * 16 + 8 + r8, a.N - 1) * a.K + piece;
  };
  auto load = [&](int j) __attribute__((always_inline)) {
    auto of = [&](const uint16_t* p) __attribute__((always_inline)) {
      const auto* q = reinterpret_cast<const rg_u32x4*>(p + line(j));
      return ONCE ? __builtin_nontemporal_load(q) : *q;
    };
    w[j][0] = of(lo);
    w[j][1] = of(hi);
    asm volatile("" ::: "memory");
  };
  rows_of(unit);
#pragma unroll
  for (int j = 0; j < P; ++j) load(j);

  const LineTurn turn_lines(lane);
  auto turn = [&](int b, const rg_u32x4& in0, const rg_u32x4& in1,
                  rg_u32x4& out0, rg_u32x4& out1)
                  __attribute__((always_inline)) {
    turn_lines(turned[wave][b & 1], in0, in1, out0, out1);
  };
#pragma unroll
  for (int j = 0; j < P; ++j)
#pragma unroll
    for (int m = 0; m < MT; ++m)
      turn(j * MT + m, xf[j][0][m], xf[j][1][m], xf[j][0][m], xf[j][1][m]);

  rg_f32x4 acc[MT];
  rg_u32x4 op[2][2];
  auto product = [&](int j) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int m = 0; m < MT; ++m)
        acc[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            __builtin_bit_cast(rg_bf16x8, op[j & 1][h]),
            __builtin_bit_cast(rg_bf16x8, xf[j][h][m]), acc[m], 0, 0, 0);
  };
  // Adds the waves' sums.  One barrier a unit: the buffer that the next unit
  // writes was read before the barrier of this one.
  int turns = 0;
  auto finish = [&](int u) __attribute__((always_inline)) {
    const int b = turns & 1;
#pragma unroll
    for (int m = 0; m < MT; ++m) sums[b][wave][m][lane] = acc[m];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    const int m = (wave - turns * MT) & (RG_WAVES - 1);   // waves take turns
    ++turns;
    if (m >= MT) return;
    rg_f32x4 y = sums[b][0][m][lane];
#pragma unroll
    for (int v = 1; v < RG_WAVES; ++v) y += sums[b][v][m][lane];
    const int row = (half * MT + m) * 16 + r16, n = u * 16 + quad * 4;
    if (row >= a.M || n >= a.N) return;
    if (a.part) {
      *reinterpret_cast<rg_f32x4*>(
          a.part + ((int64_t)split * a.M + row) * a.N + n) = y;
    } else {
      ushort4x o;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        o.v[e] = f32_to_bf16(
            y[e] + (a.bias ? bf16_to_f32(a.bias[n + e]) : 0.0f));
      *reinterpret_cast<ushort4x*>(a.out + (int64_t)row * a.N + n) = o;
    }
  };
  for (;; unit += step) {
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[m] = rg_f32x4{0.f, 0.f, 0.f, 0.f};
    if (unit + step >= units) break;
    rows_of(unit + step);
#pragma unroll
    for (int j = 0; j < P; ++j) {
      turn(j, w[j][0], w[j][1], op[j & 1][0], op[j & 1][1]);
      load(j);
      if (j) product(j - 1);
    }
    product(P - 1);
    finish(unit);
  }
#pragma unroll
  for (int j = 0; j < P; ++j) {
    turn(j, w[j][0], w[j][1], op[j & 1][0], op[j & 1][1]);
    if (j) product(j - 1);
  }
  product(P - 1);
  finish(unit);
}

// The same for 33 to 64 rows and a K in parts: three or four tiles of rows of x in
// registers, which leaves none for W, whose lines wait in LDS.
//
// A wave has a ring of R lines (16 rows of W, 128 bytes each) that fill all of the
// 160 KB that the waves' sums leave; a line goes from memory straight to its place,
// its 16-byte pieces permuted as LineTurn has them, and its place is sent for again
// as soon as it is read.  So W is streamed once, where two halves of x, in workgroups
// of their own, stream it at 4.5 TB/s.  Measured, two halves and here, with the sum of
// the parts (us, 43 and 61 rows): 4096 x 14336 30.8 32.2 and 27.4 30.9, 5120 x 17920
// 48.7 50.1 and 40.4 42.4, 5120 x 5120 18.5 19.2 and 17.6 18.5.  In one part, where W
// is short and x is most of what is loaded, it is behind (4096 x 4096 12.0 and 12.7);
// with up to 32 rows, where x leaves registers for W, too (4096 x 14336, 16 rows, 23.3
// and 25.4).
DEVINLINE rg_u32x4 rg_buffer(const uint16_t* p, int64_t bytes) {
  const uint64_t b = (uint64_t)p;
  const int n = bytes > 0x7fffffff ? 0x7fffffff : (int)bytes;
  return rg_u32x4{(uint32_t)__builtin_amdgcn_readfirstlane((int)b),
                  (uint32_t)__builtin_amdgcn_readfirstlane((int)(b >> 32)) &
                      0xffffu,
                  (uint32_t)__builtin_amdgcn_readfirstlane(n), 0x00020000u};
}

// 64 lanes x 16 bytes from memory straight to LDS, 1024 bytes from `at` on.
DEVINLINE void rg_dma(rg_u32x4 buf, int lane_off, int off, uint32_t at) {
  asm volatile(
      "s_mov_b32 m0, %0\n\ts_nop 0\n\t"
      "buffer_load_dwordx4 %1, %2, %3 offen nt lds" ::"s"(at),
      "v"(lane_off), "s"(buf), "s"(off)
      : "memory", "m0");
}

template <int P, int MT>
__global__ __launch_bounds__(64 * RG_WAVES, 2) void ring_gemm_kernel(
    RowsArgs a, int S) {
  constexpr int R = 10 - MT;
  __shared__ __attribute__((aligned(1024))) rg_u32x4 ring[RG_WAVES][R][128];
  __shared__ __attribute__((aligned(16)))
  rg_f32x4 sums[2][RG_WAVES][MT][WAVE_SIZE];
  static_assert(sizeof(ring) + sizeof(sums) == 160 * 1024);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, quad = lane >> 4, r8 = lane >> 3;
  const int split = blockIdx.x % S, step = gridDim.x / S;
  const int units = (a.N + 15) >> 4;
  int unit = blockIdx.x / S;
  if (unit >= step || unit >= units) return;

  const int k0 = (split * RG_WAVES + wave) * P * 64;
  const int rot = ((blockIdx.x >> 3) + wave) % P;
  auto line = [&](int j) __attribute__((always_inline)) {   // entries from k0 on
    return (j + rot >= P ? j + rot - P : j + rot) * 64;
  };
  // x in whole lines, all of it on its way before the first of W
  rg_u32x4 xf[P][2][MT];
#pragma unroll
  for (int j = 0; j < P; ++j)
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int m = 0; m < MT; ++m)
        xf[j][h][m] = *reinterpret_cast<const rg_u32x4*>(
            a.x + min(m * 16 + h * 8 + r8, a.M - 1) * a.x_rs + k0 + line(j) +
            (lane & 7) * 8);
  asm volatile("" ::: "memory");

  const int w0 = r8 * (a.K * 2) + ((lane & 7) ^ LineTurn::perm(r8)) * 16;
  const int w1 = (8 + r8) * (a.K * 2) + ((lane & 7) ^ LineTurn::perm(8 + r8)) * 16;
  const uint32_t lds0 =
      (uint32_t)(uintptr_t)(__attribute__((address_space(3))) rg_u32x4*)
          ring[wave];
  rg_u32x4 wbuf;
  int ahead = unit, jahead = 0, slot = 0;   // the line that is sent for next
  auto w_from = [&](int u) __attribute__((always_inline)) {
    // rows past N are zeros; past the last unit nothing is read
    const int n0 = min(u, units - 1) * 16;
    wbuf = rg_buffer(a.w + (int64_t)n0 * a.K + k0,
                     u < units ? ((int64_t)(a.N - n0) * a.K - k0) * 2 : 0);
  };
  auto send = [&]() __attribute__((always_inline)) {
    const int off = line(jahead) * 2;
    rg_dma(wbuf, w0, off, lds0 + slot * 2048);
    rg_dma(wbuf, w1, off, lds0 + slot * 2048 + 1024);
    slot = slot + 1 == R ? 0 : slot + 1;
    if (++jahead == P) {
      jahead = 0;
      ahead += step;
      w_from(ahead);
    }
  };
  w_from(unit);
#pragma unroll
  for (int i = 0; i < R; ++i) send();
  // x becomes operands in the memory of the sums
  const LineTurn turn_lines(lane);
  rg_u32x4* const scratch =
      reinterpret_cast<rg_u32x4*>(&sums[0][0][0][0]) + wave * 128;
#pragma unroll
  for (int j = 0; j < P; ++j)
#pragma unroll
    for (int m = 0; m < MT; ++m)
      turn_lines(scratch, xf[j][0][m], xf[j][1][m], xf[j][0][m], xf[j][1][m]);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");

  int used = 0, turns = 0;    // the ring's next line; units done
  for (; unit < units; unit += step, ++turns) {
    rg_f32x4 acc[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[m] = rg_f32x4{0.f, 0.f, 0.f, 0.f};
    rg_u32x4 op[2][2];
    auto product = [&](int j) __attribute__((always_inline)) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int m = 0; m < MT; ++m)
          acc[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(rg_bf16x8, op[j & 1][h]),
              __builtin_bit_cast(rg_bf16x8, xf[j][h][m]), acc[m], 0, 0, 0);
    };
#pragma unroll
    for (int j = 0; j < P; ++j) {
      // the line has arrived when at most the R - 1 behind it are under way
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * (R - 1)) : "memory");
      op[j & 1][0] = ring[wave][used][turn_lines.get];
      op[j & 1][1] = ring[wave][used][turn_lines.get_hi];
      used = used + 1 == R ? 0 : used + 1;
      if (j) product(j - 1);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      send();     // to where it was read
    }
    product(P - 1);
    // adds the waves' sums; one barrier a unit, as above
    const int b = turns & 1;
#pragma unroll
    for (int m = 0; m < MT; ++m) sums[b][wave][m][lane] = acc[m];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    const int m = (wave - turns * MT) & (RG_WAVES - 1);   // waves take turns
    if (m >= MT) continue;
    rg_f32x4 y = sums[b][0][m][lane];
#pragma unroll
    for (int v = 1; v < RG_WAVES; ++v) y += sums[b][v][m][lane];
    const int row = m * 16 + r16, n = unit * 16 + quad * 4;
    if (row < a.M && n < a.N)
      *reinterpret_cast<rg_f32x4*>(
          a.part + ((int64_t)split * a.M + row) * a.N + n) = y;
  }
  // the last pieces land in LDS that is this workgroup's until it ends
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// In how many parts K is split for M rows of x and N outputs; 0: cannot be
// taken, or would not fill the chip.
//
// A workgroup holds a compute unit (registers), so the 256 of them have to be
// evenly used: 224 workgroups take 49.0 us for 28672 x 4096 where the library
// has 54.3, 280 take 108 for 35840 x 5120 where it has 96, 160 take 47 for
// 20480 x 4096 where it has 43 (40 rows).  Splitting K to get there pays for
// the sums only over a long K: 4096 x 14336 32.2 and 39.4, but 8192 x 8192
// 33.7 and 32.8, 8192 x 4096 22.8 and 18.8.  Up to 16 rows the library is
// ahead on 128256 x 4096 (182 and 190); with the activation inside it is behind
// from 9 rows on (69 and 46).  Where both can run, rows_gemm_ahead says which.
// (These times of this kernel are from before W was loaded in whole lines, which
// took off up to a tenth; 28672 x 4096 48.2 and 54.6 since.)
int64_t rows_gemm_splits(int64_t M, int64_t N, int64_t K, bool swiglu) {
  if (M < (swiglu ? 9 : 17) || M > 64 || K < RG_BK || K % RG_BK != 0 ||
      N <= 0 || N % 4 != 0)
    return 0;
  const int64_t cols = RG_WAVES * (swiglu ? 8 : 16);
  const int64_t blocks = (N + cols - 1) / cols;
  const int64_t S = std::max<int64_t>(1, 256 / blocks);
  if (S > 1 && (swiglu || K < 3 * N || K < 6 * S * RG_BK)) return 0;
  const int64_t total = blocks * S, rounds = (total + 255) / 256;
  return total * 20 >= rounds * 256 * 17 ? S : 0;
}

// Whether rows_gemm, where it has an answer, is ahead of the library.  As one
// part it streams W at 4.9 to 5.7 TB/s whatever K is.  The library has 5.4 to
// 5.7 where rows of W do not lie a multiple of 4 KB apart, and less where they
// do (us, here and library, 33 rows: 28672 x 3072 37.9 and 36.6, 32064 x 5120
// 66.4 and 63.8; 28672 x 4096 48.2 and 54.6, 65536 x 4096 100 and 125, 28672 x
// 6144 68.7 and 80.5); over a long K it falls behind again up to 48 rows (28672
// x 11008 117 and 139, x 17920 189 and 189, at 64 rows 204 and 193, but x 11008
// 129 and 142, which the line leaves to the library).  Below 4096 this kernel's
// start and end weigh (65536 x 512 21.4 and 19.5).  A split K, where held_gemm
// does not take it, is ahead from 24 rows on and longer ones from 17 (4096 x 14080,
// 24 rows 28.3 and 39.8, as at 17 rows, which the line leaves to the library; x
// 17920 33.7 and 121).  With SwiGLU the library has a second launch and is behind
// nearly everywhere (28672 x 1024, 17 rows: 14.5 and 22.2; x 17920, 64 rows: 213 and
// 202).
bool rows_gemm_ahead(int64_t M, int64_t S, int64_t K, bool swiglu) {
  if (swiglu) return true;
  if (S > 1) return M >= 24 || K > 16384;
  return (K >= 4096 && K % 2048 == 0) || (K >= 8192 && M <= 48);
}

// out [M, N] of a product, where it is written at once
static void check_out(const torch::Tensor& out, const torch::Tensor& x,
                      int64_t N) {
  TORCH_CHECK(out.defined() && out.is_contiguous() && out.dim() == 2 &&
              out.dtype() == x.dtype() && out.size(0) == x.size(0) &&
              out.size(1) == N);
  TORCH_CHECK(out.device() == x.device(), "tensors on different devices");
}

// Writes the product to out, or, where K is in parts, returns their sums [S, M, N]
// (without the bias) and leaves out alone.
torch::Tensor rows_gemm_parts(const torch::Tensor& out, const torch::Tensor& x,
                              const torch::Tensor& w,
                              const c10::optional<torch::Tensor>& bias,
                              int64_t gate) {
  const bool swiglu = gate != 0;
  TORCH_CHECK(gate >= 0 && gate <= 2);
  TORCH_CHECK(x.is_cuda() && x.dim() == 2 && x.stride(1) == 1 &&
              x.dtype() == torch::kBFloat16 && w.dtype() == x.dtype() &&
              w.dim() == 2 && w.is_contiguous());
  const int64_t M = x.size(0), K = x.size(1);
  const int64_t N = swiglu ? w.size(0) / 2 : w.size(0);
  const int64_t S = rows_gemm_splits(M, N, K, swiglu);
  TORCH_CHECK(S >= 1);
  if (S == 1) check_out(out, x, N);
  TORCH_CHECK(w.size(1) == K && w.size(0) == (swiglu ? 2 * N : N) &&
              x.stride(0) % 8 == 0);
  TORCH_CHECK(w.device() == x.device(), "tensors on different devices");
  TORCH_CHECK((reinterpret_cast<uintptr_t>(x.data_ptr()) & 15) == 0 &&
              (reinterpret_cast<uintptr_t>(w.data_ptr()) & 15) == 0);
  if (bias.has_value())
    TORCH_CHECK(!swiglu && bias->dtype() == x.dtype() &&
                bias->device() == x.device() && bias->is_contiguous() &&
                bias->numel() == N);
  const at::cuda::CUDAGuard guard(x.device());
  hipStream_t stream = at::cuda::getCurrentCUDAStream();
  const int64_t cols = RG_WAVES * (swiglu ? 8 : 16);
  const int64_t blocks = (N + cols - 1) / cols;
  torch::Tensor part;
  if (S > 1)
    part = torch::empty({S, M, N}, x.options().dtype(torch::kFloat32));
  RowsArgs a{S > 1 ? nullptr : (uint16_t*)out.data_ptr(),
             S > 1 ? part.data_ptr<float>() : nullptr,
             (const uint16_t*)x.data_ptr(),
             (const uint16_t*)w.data_ptr(),
             bias.has_value() ? (const uint16_t*)bias->data_ptr() : nullptr,
             (int)M, (int)N, (int)K, x.stride(0)};
  const dim3 grid(blocks, S);
  const bool once = K >= RG_ONCE;
#define LAUNCH_RG(...)                                                       \
  hipLaunchKernelGGL((rows_gemm_kernel<__VA_ARGS__>), grid,                  \
                     dim3(64 * RG_WAVES), 0, stream, a)
#define LAUNCH_RG_G(MT, ONCE)                                                \
  do {                                                                       \
    if (gate == 2) LAUNCH_RG(MT, 2, ONCE);                                   \
    else if (gate == 1) LAUNCH_RG(MT, 1, ONCE);                              \
    else LAUNCH_RG(MT, 0, ONCE);                                             \
  } while (0)
#define LAUNCH_RG_M(MT)                                                      \
  do {                                                                       \
    if (once) LAUNCH_RG_G(MT, true);                                         \
    else LAUNCH_RG_G(MT, false);                                             \
  } while (0)
  if (M <= 16 && gate == 2 && once) LAUNCH_RG(1, 2, true);   // with a gate only
  else if (M <= 16 && gate == 2) LAUNCH_RG(1, 2, false);
  else if (M <= 16 && once) LAUNCH_RG(1, 1, true);
  else if (M <= 16) LAUNCH_RG(1, 1, false);
  else if (M <= 32) LAUNCH_RG_M(2);
  else if (M <= 48) LAUNCH_RG_M(3);
  else LAUNCH_RG_G(4, false);
#undef LAUNCH_RG_M
#undef LAUNCH_RG_G
#undef LAUNCH_RG
  HIP_CHECK_KERNEL();
  return part;
}

void rows_gemm(torch::Tensor out, torch::Tensor x, torch::Tensor w,
               c10::optional<torch::Tensor> bias, int64_t gate) {
  check_out(out, x, gate != 0 ? w.size(0) / 2 : w.size(0));
  const auto part = rows_gemm_parts(out, x, w, bias, gate);
  if (part.defined()) sum_parts(out, part, bias);
}

// Whether ring_gemm takes a held product whose K is in parts.  It streams W once, but a
// workgroup's start, with all of x, is longer than that of two halves, and few outputs
// share it (us, two halves and ring_gemm, 43 and 61 rows or 64: 1024 x 5120 8.9 9.1 and
// 10.0 10.6, 2560 x 6144 13.4 14.2 and 14.1 15.3, 3072 x 8192 16.5 18.1 and 17.5 18.3,
// 1536 x 10240 13.0 13.8 and 13.4 14.6; 4096 x 6144 16.0 16.8 and 15.5 17.1, 2048 x 10240
// 15.0 15.8 and 14.4 15.3, 1024 x 12288 13.9 15.1 and 13.2 13.9, 4096 x 14336 30.2 31.5
// and 26.3 29.9).
static bool ring_takes(int64_t M, int64_t N, int64_t K) {
  const int64_t least = K >= 12288   ? 1024
                        : K >= 10240 ? 2048
                        : M <= 48    ? 4096
                                     : 5120;
  return M > 32 && N >= least;
}

// In how many parts held_gemm cuts K (a wave's part is four to eight lines of
// 64 entries); 0: it cannot.
int64_t held_splits(int64_t M, int64_t N, int64_t K) {
  if (M < 1 || M > 64 || N < 1 || N % 4 != 0 || N > (1 << 26) ||
      K > (1 << 20))
    return 0;
  // four tiles of rows leave registers for six lines, where it can be had so
  for (const int64_t most : {M > 48 && ring_takes(M, N, K) ? 6 : 8, 8})
    for (int64_t S = 1; S <= 8; ++S)
      if (K % (RG_WAVES * 64 * S) == 0) {
        const int64_t lines = K / (RG_WAVES * 64 * S);
        if (lines >= 4 && lines <= (S == 1 ? 8 : most)) return S;
      }
  return 0;
}

// Whether held_gemm is ahead of the library (and of rows_gemm in parts); gemv
// has up to six rows, rows_gemm what it takes whole (us, library and here).  With
// one part, up to 32 rows, at all 60 measured sizes of 16 x 2048 to 10240 x 4096
// (16 x 2048 5.2 and 3.3, 10240 x 4096 23.4 and 20.2), wider ones to 16 rows
// (20480 x 4096 75.6 and 37.2, 32000 x 3584 46.1 and 41.2), to 32 from K = 2560 on
// (20480 x 3584 40.9 and 31.3, but 32000 x 3584 41.4 and 43.1, 16384 x 2048 17.3 and
// 18.6).  At a vocabulary's width it is ahead since its loads are nontemporal: 128256
// x 4096, 8 and 16 rows, 190 183 and 169 171 (narrow_gemm, asked first, takes those
// from K = 4096 on).
// The two halves of more rows stream W at 4.5 TB/s: 10240 x 3584, 64 rows, 25.0 and
// 22.3, 16384 x 3584 30.4 and 38.2.  Parts cost their sums, and a short K the
// library has tiles for: up to 32 rows 10240 x 5120 33.2 and 27.5, 16384 x 5120 37.6
// and 39.6, 256 x 8192 8.8 and 9.2; of 64 rows 6144 x 14336 63.6 and 58.4, 8192 x
// 8192 34.5 and 36.3.  In two parts (1024 to 8192 x 5120 to 8192, 7 to 32 rows, 288
// sizes) it takes 0.47 to 1.0 of the library's time, but around 16 rows of 2560 x
// 5120 to 8192 and 3072 x 6144, and for 4096 x 7168 and 8192, 6144 x 8192 and 8192 x
// 5120, where it is 2 to 8 % behind (4096 x 8192, 16 rows, 16.9 and 17.9; 5120 x 8192,
// 17 rows, 25.9 and 21.8).
static bool held_ahead(int64_t M, int64_t N, int64_t K, int64_t S) {
  if (M < 7) return false;
  if (M > 32) return S == 1 ? N <= 10240 : N >= 1024 && N <= 6144;
  if (S == 1)
    return N <= 10240 ||
           (M <= 16 ? N <= 32768 || N >= 65536 : K >= 2560 && N <= 20480);
  return N <= 10240 && (M <= 16 || N >= 1024);
}

bool held_gemm_takes(int64_t M, int64_t N, int64_t K) {
  const int64_t S = held_splits(M, N, K);
  return S > 0 && held_ahead(M, N, K, S) &&
         !(rows_gemm_splits(M, N, K, false) == 1 &&
           rows_gemm_ahead(M, 1, K, false));
}

// The same with x in registers.
torch::Tensor held_gemm_parts(const torch::Tensor& out, const torch::Tensor& x,
                              const torch::Tensor& w,
                              const c10::optional<torch::Tensor>& bias) {
  TORCH_CHECK(x.is_cuda() && x.dim() == 2 && x.stride(1) == 1 &&
              x.dtype() == torch::kBFloat16 && w.dtype() == x.dtype() &&
              w.dim() == 2 && w.is_contiguous());
  const int64_t M = x.size(0), K = x.size(1), N = w.size(0);
  const int64_t S = held_splits(M, N, K);
  TORCH_CHECK(S >= 1);
  if (S == 1) check_out(out, x, N);
  TORCH_CHECK(w.size(1) == K && x.stride(0) % 8 == 0);
  TORCH_CHECK(w.device() == x.device(), "tensors on different devices");
  TORCH_CHECK((reinterpret_cast<uintptr_t>(x.data_ptr()) & 15) == 0 &&
              (reinterpret_cast<uintptr_t>(w.data_ptr()) & 15) == 0);
  if (bias.has_value())
    TORCH_CHECK(bias->dtype() == x.dtype() && bias->device() == x.device() &&
                bias->is_contiguous() && bias->numel() == N);
  const at::cuda::CUDAGuard guard(x.device());
  hipStream_t stream = at::cuda::getCurrentCUDAStream();
  torch::Tensor part;
  if (S > 1)
    part = torch::empty({S, M, N}, x.options().dtype(torch::kFloat32));
  RowsArgs a{S > 1 ? nullptr : (uint16_t*)out.data_ptr(),
             S > 1 ? part.data_ptr<float>() : nullptr,
             (const uint16_t*)x.data_ptr(),
             (const uint16_t*)w.data_ptr(),
             bias.has_value() ? (const uint16_t*)bias->data_ptr() : nullptr,
             (int)M, (int)N, (int)K, x.stride(0)};
  const bool once = M <= 32 && N * K >= HELD_ONCE;
  const int64_t lines = K / (RG_WAVES * 64 * S);
#define LAUNCH_RING(P, MT)                                                    \
  case MT * 16 + P:                                                           \
    hipLaunchKernelGGL((ring_gemm_kernel<P, MT>), dim3(256),                  \
                       dim3(64 * RG_WAVES), 0, stream, a, (int)S);            \
    break
  if (S > 1 && ring_takes(M, N, K) && (M <= 48 || lines <= 6)) {
    switch ((M > 48 ? 4 : 3) * 16 + lines) {   // four lines only of four tiles
      LAUNCH_RING(5, 3);
      LAUNCH_RING(6, 3);
      LAUNCH_RING(7, 3);
      LAUNCH_RING(8, 3);
      LAUNCH_RING(4, 4);
      LAUNCH_RING(5, 4);
      LAUNCH_RING(6, 4);
      default: TORCH_CHECK(false, "no such parts: ", lines);
    }
    HIP_CHECK_KERNEL();
    return part;
  }
#undef LAUNCH_RING
#define LAUNCH_HELD_AS(...)                                                   \
  hipLaunchKernelGGL((held_gemm_kernel<__VA_ARGS__>), dim3(256),              \
                     dim3(64 * RG_WAVES), 0, stream, a, (int)S)
#define LAUNCH_HELD(P)                                                        \
  case P:                                                                     \
    if (M > 32) LAUNCH_HELD_AS(P, 2, 2, false);                               \
    else if (M > 16 && once) LAUNCH_HELD_AS(P, 2, 1, true);                   \
    else if (M > 16) LAUNCH_HELD_AS(P, 2, 1, false);                          \
    else if (once) LAUNCH_HELD_AS(P, 1, 1, true);                             \
    else LAUNCH_HELD_AS(P, 1, 1, false);                                      \
    break
  switch (lines) {
    LAUNCH_HELD(4);
    LAUNCH_HELD(5);
    LAUNCH_HELD(6);
    LAUNCH_HELD(7);
    LAUNCH_HELD(8);
  }
#undef LAUNCH_HELD
#undef LAUNCH_HELD_AS
  HIP_CHECK_KERNEL();
  return part;
}

void held_gemm(torch::Tensor out, torch::Tensor x, torch::Tensor w,
               c10::optional<torch::Tensor> bias) {
  check_out(out, x, w.size(0));
  const auto part = held_gemm_parts(out, x, w, bias);
  if (part.defined()) sum_parts(out, part, bias);
}

}  // namespace igw
