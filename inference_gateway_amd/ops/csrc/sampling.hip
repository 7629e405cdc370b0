// Fused top-k / top-p / temperature sampling kernel for gfx950.
//
// Net-new engine scope (SURVEY.md §7 stage 3b). One workgroup per sequence,
// operating on the fp32 logits row (vocab ~128k):
//
//   1. block max M in one pass;
//   2. greedy path (temperature == 0): argmax with lowest-index tie break;
//   3. joint 4-level radix walk over the monotone uint32 key image of the
//      fp32 logit: each level is ONE pass that builds a count histogram
//      (for the top-k threshold) and an exp-weighted histogram (for the
//      top-p mass threshold) simultaneously, into WAVE-PRIVATE LDS bins
//      (logit exponents cluster in a handful of bins, so shared-bin atomics
//      would serialize across the whole block); Z falls out of level 3's
//      weight histogram for free;
//   4. kept-mass pass, then an inverse-CDF walk over the kept set in index
//      order with the caller-supplied uniform u (host draws it from torch's
//      RNG so runs are reproducible under torch.manual_seed).
//
// Thresholds are VALUE thresholds: top-k keeps ties of the k-th value; the
// nucleus set is the smallest value-threshold set with mass >= p*Z. The
// Python reference (ops/torch_ref.py::sample_ref) implements exactly these
// semantics, so GPU vs CPU tests compare token-for-token with fixed u.

#include <ATen/cuda/CUDAContext.h>
#include <torch/extension.h>

#include <climits>

#include "common.h"

namespace igw {

DEVINLINE uint32_t f32_key(float x) {
  union {
    float f;
    uint32_t u;
  } v;
  v.f = x;
  return (v.u & 0x80000000u) ? ~v.u : (v.u | 0x80000000u);
}

template <int BLOCK>
__global__ __launch_bounds__(BLOCK) void sample_kernel(
    int32_t* __restrict__ out,            // [B]
    const float* __restrict__ logits,     // [B, V]
    const float* __restrict__ temperature,// [B]
    const int32_t* __restrict__ top_k,    // [B] (<=0 => disabled)
    const float* __restrict__ top_p,      // [B] (>=1 => disabled)
    const float* __restrict__ uniforms,   // [B]
    int V) {
  constexpr int NW = BLOCK / WAVE_SIZE;
  __shared__ float redf[NW];
  __shared__ uint32_t ubins[NW][256];
  __shared__ float fbins[NW][256];
  __shared__ uint32_t s_u32[2];
  __shared__ float s_f32[4];
  __shared__ float seg_sums[BLOCK + 1];

  const int seq = blockIdx.x;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const float* row = logits + (int64_t)seq * V;
  const float temp = temperature[seq];
  const bool greedy = (temp <= 0.0f);
  const float inv_t = greedy ? 1.0f : 1.0f / temp;

  // ---- pass 1: max ----
  float mx = -INFINITY;
  for (int i = tid; i < V; i += BLOCK) mx = fmaxf(mx, row[i] * inv_t);
  mx = wave_reduce_max(mx);
  if (lane == 0) redf[wave] = mx;
  __syncthreads();
  if (tid == 0) {
    float r = redf[0];
    for (int w = 1; w < NW; ++w) r = fmaxf(r, redf[w]);
    s_f32[0] = r;
  }
  __syncthreads();
  const float M = s_f32[0];

  if (greedy) {
    if (tid == 0) s_u32[0] = 0xffffffffu;
    __syncthreads();
    for (int i = tid; i < V; i += BLOCK) {
      if (row[i] == M) atomicMin(&s_u32[0], (uint32_t)i);
    }
    __syncthreads();
    if (tid == 0) out[seq] = (int32_t)s_u32[0];
    return;
  }

  const int k = top_k[seq];
  const float p = top_p[seq];
  const bool do_k = (k > 0 && k < V);
  const bool do_p = (p < 1.0f);

  // ---- joint radix walk: 4 levels, one pass each ----
  uint32_t tk_prefix = 0, tp_prefix = 0;
  uint32_t tk_remaining = do_k ? (uint32_t)k : 0;
  float tp_target = 0.0f;  // set after level 3 (needs Z)
  float Z = 0.0f;

  for (int level = 3; level >= 0; --level) {
    for (int b = tid; b < 256; b += BLOCK) {
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        ubins[w][b] = 0;
        fbins[w][b] = 0.0f;
      }
    }
    __syncthreads();
    const int shift = level * 8;
    for (int i = tid; i < V; i += BLOCK) {
      const float x = row[i] * inv_t;
      const uint32_t key = f32_key(x);
      const uint32_t hi = (level == 3) ? 0 : (key >> (shift + 8));
      const uint32_t b = (key >> shift) & 0xff;
      if (do_k && (level == 3 || hi == tk_prefix)) {
        atomicAdd(&ubins[wave][b], 1u);
      }
      if (level == 3 || hi == tp_prefix) {
        // level 3 weight histogram doubles as Z (do_p or not)
        atomicAdd(&fbins[wave][b], __expf(x - M));
      }
    }
    __syncthreads();
    if (tid == 0) {
      if (level == 3) {
        float z = 0.0f;
        for (int b = 0; b < 256; ++b)
          for (int w = 0; w < NW; ++w) z += fbins[w][b];
        Z = z;
        s_f32[1] = z;
        tp_target = p * z;
      }
      if (do_k) {
        uint32_t cum = 0;
        int bstar = 0;
        for (int b = 255; b >= 0; --b) {
          uint32_t c = 0;
          for (int w = 0; w < NW; ++w) c += ubins[w][b];
          if (cum + c >= tk_remaining) {
            bstar = b;
            break;
          }
          cum += c;
        }
        tk_prefix = (tk_prefix << 8) | (uint32_t)bstar;
        tk_remaining -= cum;
        s_u32[0] = tk_prefix;
      }
      if (do_p) {
        float cum = 0.0f;
        int bstar = 0;
        for (int b = 255; b >= 0; --b) {
          float c = 0.0f;
          for (int w = 0; w < NW; ++w) c += fbins[w][b];
          if (cum + c >= tp_target) {
            bstar = b;
            break;
          }
          cum += c;
        }
        tp_prefix = (tp_prefix << 8) | (uint32_t)bstar;
        tp_target -= cum;
        s_f32[2] = tp_target;
        s_u32[1] = tp_prefix;
      }
    }
    __syncthreads();
    if (do_k) tk_prefix = s_u32[0];
    if (do_p) {
      tp_prefix = s_u32[1];
      tp_target = s_f32[2];
    }
    // each thread needs tk_remaining only on thread 0; prefixes broadcast
    if (!do_k && !do_p && level == 3) break;  // pure-temperature sampling
  }

  const uint32_t tau =
      max(do_k ? tk_prefix : 0u, do_p ? tp_prefix : 0u);

  // ---- kept mass + per-thread segment sums (one fused pass) ----
  const int seg = (V + BLOCK - 1) / BLOCK;
  const int s0 = tid * seg;
  const int s1 = min(V, s0 + seg);
  float segsum = 0.0f;
  for (int i = s0; i < s1; ++i) {
    const float x = row[i] * inv_t;
    if (f32_key(x) >= tau) segsum += __expf(x - M);
  }
  seg_sums[tid] = segsum;
  __syncthreads();
  if (tid == 0) {
    float run = 0.0f;
    for (int t = 0; t < BLOCK; ++t) {
      const float s = seg_sums[t];
      seg_sums[t] = run;
      run += s;
    }
    seg_sums[BLOCK] = run;  // = Zf
    s_u32[0] = 0xffffffffu;
  }
  __syncthreads();

  // ---- inverse-CDF walk in index order ----
  const float zf = seg_sums[BLOCK];
  const float target = uniforms[seq] * zf;
  const float base = seg_sums[tid];
  const float next = seg_sums[tid + 1];
  if (target >= base && (target < next || tid == BLOCK - 1)) {
    float run = base;
    int chosen = -1;
    for (int i = s0; i < s1; ++i) {
      const float x = row[i] * inv_t;
      if (f32_key(x) >= tau) {
        run += __expf(x - M);
        chosen = i;
        if (run > target) break;
      }
    }
    if (chosen >= 0) atomicMin(&s_u32[0], (uint32_t)chosen);
  }
  __syncthreads();
  if (tid == 0) {
    uint32_t c = s_u32[0];
    if (c == 0xffffffffu) {
      // numeric corner (u ~ 1.0): fall back to argmax
      c = 0;
      float best = -INFINITY;
      for (int i = 0; i < V; ++i) {
        const float x = row[i] * inv_t;
        if (x > best) {
          best = x;
          c = i;
        }
      }
    }
    out[seq] = (int32_t)c;
  }
}

// ---------------------------------------------------------------------------
// bf16 fast path.  The lm_head emits bf16; sampling directly on the bf16
// bits (a) halves the logits traffic vs the fp32 path and (b) shrinks the
// monotone key to 16 bits, so the radix walk is 2 levels instead of 4.
// Thresholds are found on the UNSCALED bf16 key (temperature > 0 preserves
// order); only the exp-weights use the temperature.  Loads are uint4
// (8 bf16/lane), and per-8 runs of equal bins are merged before the LDS
// atomic — with near-flat random-init logits the bins collide wave-wide,
// which is what made the fp32 kernel's histogram passes serialize
// (profiles/r01: 1.48 ms at B=512).
// ---------------------------------------------------------------------------

DEVINLINE uint32_t bf16_key(uint16_t u) {
  return (u & 0x8000u) ? (uint32_t)(~u & 0xffffu) : (uint32_t)(u | 0x8000u);
}

DEVINLINE float bf16_val(uint16_t u) {
  union {
    uint32_t q;
    float f;
  } v;
  v.q = ((uint32_t)u) << 16;
  return v.f;
}

// Parallel suffix-threshold search over 256 combined bins, run by ONE wave.
// vals: combined per-bin values (descending walk from bin 255).  Returns
// (bstar, remaining) through s_res: the first bin b (from the top) where
// cum_above + vals[b] >= target, with remaining = target - cum_above.
template <typename T>
DEVINLINE void suffix_threshold_search(const T* vals, T target, int lane,
                                       uint32_t* s_b, T* s_rem) {
  T lsum = T(0);
#pragma unroll
  for (int j = 0; j < 4; ++j) lsum += vals[lane * 4 + j];
  // inclusive suffix sum across lanes: s[l] = sum_{l' >= l} lsum[l']
  T s = lsum;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const T t = __shfl_down(s, off, 64);
    if (lane + off < 64) s += t;
  }
  const T above = s - lsum;  // bins owned by lanes > l
  if (s >= target && (lane == 63 || above < target)) {
    // descend within this lane's 4 bins, highest first
    T cum = above;
    int bstar = lane * 4;
    T rem = target - cum;
#pragma unroll
    for (int j = 3; j >= 0; --j) {
      const int b = lane * 4 + j;
      const T c = vals[b];
      if (cum + c >= target) {
        bstar = b;
        rem = target - cum;
        break;
      }
      cum += c;
    }
    *s_b = (uint32_t)bstar;
    *s_rem = rem;
  }
  // degenerate: target exceeds the total (float rounding at p ~ 1.0) —
  // fall through to bin 0 like the serial walk
  if (lane == 0 && s < target) {
    *s_b = 0;
    *s_rem = target - s;
  }
}

template <int BLOCK>
__global__ __launch_bounds__(BLOCK) void sample_bf16_kernel(
    int32_t* __restrict__ out,             // [B]
    const uint16_t* __restrict__ logits,   // [B, V] bf16 bits
    const float* __restrict__ temperature, // [B]
    const int32_t* __restrict__ top_k,     // [B] (<=0 => disabled)
    const float* __restrict__ top_p,       // [B] (>=1 => disabled)
    const float* __restrict__ uniforms,    // [B]
    int V) {
  constexpr int NW = BLOCK / WAVE_SIZE;
  constexpr int REP = 2;  // bin replicas per wave (LDS-atomic conflict
                          // width vs footprint). Measured: REP=2 (~36 KB,
                          // 4 blocks/CU) == REP=4 (~68 KB, 2 blocks/CU)
                          // at B=512 — the histogram passes are
                          // per-element VALU-bound, not LDS- or
                          // occupancy-bound; keep the smaller footprint
  __shared__ float redf[NW];
  __shared__ uint32_t ubins[NW][REP][256];
  __shared__ float fbins[NW][REP][256];
  __shared__ uint32_t ucomb[256];
  __shared__ float fcomb[256];
  __shared__ uint32_t s_u32[4];
  __shared__ float s_f32[4];
  __shared__ float seg_sums[BLOCK + 1];

  const int seq = blockIdx.x;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const uint16_t* row = logits + (int64_t)seq * V;
  const float temp = temperature[seq];
  const bool greedy = (temp <= 0.0f);
  const float inv_t = greedy ? 1.0f : 1.0f / temp;
  const int V8 = V >> 3;
  const uint4* row8 = reinterpret_cast<const uint4*>(row);

  // ---- pass 1: unscaled max (order == scaled order) ----
  float mx = -INFINITY;
  for (int i = tid; i < V8; i += BLOCK) {
    const uint4 v = row8[i];
#pragma unroll
    for (int h = 0; h < 4; ++h) {
      const uint32_t q = (&v.x)[h];
      mx = fmaxf(mx, bf16_val((uint16_t)(q & 0xffffu)));
      mx = fmaxf(mx, bf16_val((uint16_t)(q >> 16)));
    }
  }
  for (int i = (V8 << 3) + tid; i < V; i += BLOCK)
    mx = fmaxf(mx, bf16_val(row[i]));
  mx = wave_reduce_max(mx);
  if (lane == 0) redf[wave] = mx;
  __syncthreads();
  if (tid == 0) {
    float r = redf[0];
    for (int w = 1; w < NW; ++w) r = fmaxf(r, redf[w]);
    s_f32[0] = r;
  }
  __syncthreads();
  const float M = s_f32[0];

  if (greedy) {
    if (tid == 0) s_u32[0] = 0xffffffffu;
    __syncthreads();
    for (int i = tid; i < V; i += BLOCK) {
      if (bf16_val(row[i]) == M) atomicMin(&s_u32[0], (uint32_t)i);
    }
    __syncthreads();
    if (tid == 0) out[seq] = (int32_t)s_u32[0];
    return;
  }

  const int k = top_k[seq];
  const float p = top_p[seq];
  const bool do_k = (k > 0 && k < V);
  const bool do_p = (p < 1.0f);
  uint32_t tau = 0;

  if (do_k || do_p) {
    uint32_t tk_prefix = 0, tp_prefix = 0;
    uint32_t tk_remaining = do_k ? (uint32_t)k : 0;
    float tp_target = 0.0f;
    const int rep = (lane >> 3) & (REP - 1);

    for (int level = 1; level >= 0; --level) {
      for (int b = tid; b < 256; b += BLOCK) {
#pragma unroll
        for (int w = 0; w < NW; ++w)
#pragma unroll
          for (int r = 0; r < REP; ++r) {
            ubins[w][r][b] = 0;
            fbins[w][r][b] = 0.0f;
          }
      }
      __syncthreads();
      const int shift = level * 8;
      uint32_t* const my_u = ubins[wave][rep];
      float* const my_f = fbins[wave][rep];
      // run-merge accumulators live across the WHOLE pass: near-flat
      // logits keep hitting the same bin, so each thread issues only a
      // handful of LDS atomics instead of one per 8 elements
      uint32_t runb_k = 0xffffffffu, runc_k = 0;
      uint32_t runb_p = 0xffffffffu;
      float runw_p = 0.0f;
      for (int i = tid; i < V8; i += BLOCK) {
        const uint4 v = row8[i];
#pragma unroll
        for (int h = 0; h < 8; ++h) {
          const uint32_t q = (&v.x)[h >> 1];
          const uint16_t u = (uint16_t)((h & 1) ? (q >> 16) : (q & 0xffffu));
          const uint32_t key = bf16_key(u);
          const uint32_t hi = (level == 1) ? 0 : (key >> 8);
          const uint32_t b = (key >> shift) & 0xff;
          if (do_k && (level == 1 || hi == tk_prefix)) {
            if (b == runb_k) {
              ++runc_k;
            } else {
              if (runc_k) atomicAdd(&my_u[runb_k], runc_k);
              runb_k = b;
              runc_k = 1;
            }
          }
          if (level == 1 || hi == tp_prefix) {
            const float w = __expf((bf16_val(u) - M) * inv_t);
            if (b == runb_p) {
              runw_p += w;
            } else {
              if (runb_p != 0xffffffffu) atomicAdd(&my_f[runb_p], runw_p);
              runb_p = b;
              runw_p = w;
            }
          }
        }
      }
      if (runc_k) atomicAdd(&my_u[runb_k], runc_k);
      if (runb_p != 0xffffffffu) atomicAdd(&my_f[runb_p], runw_p);
      for (int i = (V8 << 3) + tid; i < V; i += BLOCK) {
        const uint16_t u = row[i];
        const uint32_t key = bf16_key(u);
        const uint32_t hi = (level == 1) ? 0 : (key >> 8);
        const uint32_t b = (key >> shift) & 0xff;
        if (do_k && (level == 1 || hi == tk_prefix))
          atomicAdd(&my_u[b], 1u);
        if (level == 1 || hi == tp_prefix)
          atomicAdd(&my_f[b], __expf((bf16_val(u) - M) * inv_t));
      }
      __syncthreads();
      // combine replicas (parallel: one thread per bin)
      for (int b = tid; b < 256; b += BLOCK) {
        uint32_t cu = 0;
        float cf = 0.0f;
#pragma unroll
        for (int w = 0; w < NW; ++w)
#pragma unroll
          for (int r = 0; r < REP; ++r) {
            cu += ubins[w][r][b];
            cf += fbins[w][r][b];
          }
        ucomb[b] = cu;
        fcomb[b] = cf;
      }
      __syncthreads();
      if (level == 1) {
        // Z = sum of the weight bins (parallel block reduce)
        float z = (tid < 256) ? fcomb[tid] : 0.0f;
        z = wave_reduce_sum(z);
        if (lane == 0) redf[wave] = z;
        __syncthreads();
        if (tid == 0) {
          float zz = 0.0f;
          for (int w = 0; w < NW; ++w) zz += redf[w];
          s_f32[1] = zz;
        }
        __syncthreads();
        if (do_p) tp_target = p * s_f32[1];
      }
      // wave 0: top-k count search; wave 1: top-p mass search
      if (do_k && wave == 0) {
        suffix_threshold_search<uint32_t>(ucomb, tk_remaining, lane,
                                          &s_u32[0], &s_u32[1]);
      }
      if (do_p && wave == (NW > 1 ? 1 : 0)) {
        suffix_threshold_search<float>(fcomb, tp_target, lane, &s_u32[2],
                                       &s_f32[2]);
      }
      __syncthreads();
      if (do_k) {
        tk_prefix = (tk_prefix << 8) | (s_u32[0] & 0xffu);
        tk_remaining = s_u32[1];
      }
      if (do_p) {
        tp_prefix = (tp_prefix << 8) | (s_u32[2] & 0xffu);
        tp_target = s_f32[2];
      }
      __syncthreads();
    }
    tau = max(do_k ? tk_prefix : 0u, do_p ? tp_prefix : 0u);
  }

  // ---- kept mass + per-thread segment sums (one fused pass,
  //      vectorized uint4 loads; segments 8-aligned) ----
  const int seg = (((V + BLOCK - 1) / BLOCK) + 7) & ~7;
  const int s0 = min(V, tid * seg);
  const int s1 = min(V, s0 + seg);
  float segsum = 0.0f;
  int i = s0;
  for (; i + 8 <= s1; i += 8) {
    const uint4 v = *reinterpret_cast<const uint4*>(row + i);
#pragma unroll
    for (int h = 0; h < 8; ++h) {
      const uint32_t q = (&v.x)[h >> 1];
      const uint16_t u = (uint16_t)((h & 1) ? (q >> 16) : (q & 0xffffu));
      if (bf16_key(u) >= tau)
        segsum += __expf((bf16_val(u) - M) * inv_t);
    }
  }
  for (; i < s1; ++i) {
    const uint16_t u = row[i];
    if (bf16_key(u) >= tau) segsum += __expf((bf16_val(u) - M) * inv_t);
  }
  seg_sums[tid] = segsum;
  __syncthreads();
  if (tid == 0) {
    float run = 0.0f;
    for (int t = 0; t < BLOCK; ++t) {
      const float s = seg_sums[t];
      seg_sums[t] = run;
      run += s;
    }
    seg_sums[BLOCK] = run;  // = Zf
    s_u32[0] = 0xffffffffu;
  }
  __syncthreads();

  // ---- inverse-CDF walk in index order ----
  const float zf = seg_sums[BLOCK];
  const float target = uniforms[seq] * zf;
  const float base = seg_sums[tid];
  const float next = seg_sums[tid + 1];
  if (target >= base && (target < next || tid == BLOCK - 1)) {
    float run = base;
    int chosen = -1;
    for (int i = s0; i < s1; ++i) {
      const uint16_t u = row[i];
      if (bf16_key(u) >= tau) {
        run += __expf((bf16_val(u) - M) * inv_t);
        chosen = i;
        if (run > target) break;
      }
    }
    if (chosen >= 0) atomicMin(&s_u32[0], (uint32_t)chosen);
  }
  __syncthreads();
  if (tid == 0) {
    uint32_t c = s_u32[0];
    if (c == 0xffffffffu) {
      // numeric corner (u ~ 1.0): fall back to argmax
      c = 0;
      float best = -INFINITY;
      for (int i = 0; i < V; ++i) {
        const float x = bf16_val(row[i]);
        if (x > best) {
          best = x;
          c = i;
        }
      }
    }
    out[seq] = (int32_t)c;
  }
}

// ---------------------------------------------------------------------------
// bf16 rows that fit a workgroup's registers (V <= 8 * 512 * NCH): the row is
// read ONCE, 16 bytes a load, past the memory side's cache, and every further pass
// runs on registers.
//
//   1. maximum, and for top-p the total mass Z;
//      From there the row is kept as keys, whose order is the logits', so that
//      the largest of a chunk of eight takes a few packed instructions and a
//      wave goes past the chunks that no lane needs;
//   2. thresholds: counts per exact bf16 value in LDS for the keys from the
//      top down, first the 128 keys (an octave) below the maximum, then the 256
//      after them, then windows of 4096, each starting at the highest key that
//      is left.  The mass of a value is count * exp, so no exponential is taken
//      per element here.  The first window that holds either threshold decides:
//      the other one is lower and max(tau_k, tau_p) is wanted.  With more than
//      eight chunks a thread, those with a key of the first window (commonly a
//      few hundred of 8192) go to a list in LDS, and counts and draw are loops
//      over it;
//   3. the draw: listed chunks with a kept element, if they are at most as many
//      as threads, are put in index order by counting, and one running sum finds
//      the chunk.  Otherwise kept mass per (chunk, wave) cell in index order,
//      cells without a kept element skipped; the cell, the lane, the element.
//
// Bound: the row's 64 KB to 128 KB arrive at HBM speed, then come passes over all its
// elements on the vector units, one for the mass, one for the keys and one for
// every window or cell pass that is needed, with two to four rows on a compute unit;
// with the passes written out for up to 16 chunks also the 64 KB instruction
// cache, which is why what is rare is a loop.  Each of the four passes of
// sample_bf16_kernel reads the row again and updates LDS bins for all elements.
// 1024 rows of 32064, greedy / top-k 50 and top-p / top-p 0.9 / top-k 40 / no
// limits: 12.8, 36, 43, 29 and 22.5 us; with elements instead of keys, every pass
// over all of them and the list's work in the cells 14.4, 39, 65, 33 and 28
// (the list there: 15, 38, 47, 35 and 26, hence the line at eight chunks).
// Rows of more than 8 * 512 * 16 logits go to sample_bf16_stream_kernel: they leave
// registers for one row a compute unit only.  Those of up to 4096 keep
// sample_bf16_kernel, where its passes are short (1000 logits, 300 rows, greedy /
// top-k and top-p / top-p: 3.0, 15.9 and 15.0 us, here 7.5, 17.0 and 28.3 before;
// 4099 logits 3.9, 27.0 and 24.7, here 3.8, 10.9 and 17.7).  There are as many sizes of the kernel as
// keep rows without limits ahead of that one, which has few passes for them (300
// rows of 33000 29.7 us, here 35.3 with 16 chunks, 20.5 with 12).
// ---------------------------------------------------------------------------
constexpr int SR_THREADS = 512;
constexpr int SR_WAVES = SR_THREADS / WAVE_SIZE;
constexpr int SR_FIRST = 128;    // keys of the first window
constexpr int SR_SECOND = 256;   // of the second
constexpr int SR_WINDOW = 4096;  // of the others
constexpr int SR_LIST = 2048;    // chunks of the first window that are listed

// Sums, maxima and running sums over the wave by lane exchanges of the vector
// units (one through LDS takes six round trips).  A lane without a partner gets
// `none`.
template <int CTRL, int ROWS = 0xf, class T>
DEVINLINE T sr_lane(T x, T none) {
  return __builtin_bit_cast(
      T, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, none),
                                     __builtin_bit_cast(int, x), CTRL, ROWS,
                                     0xf, false));
}
DEVINLINE void sr_both16(float x, float& a, float& b) {
  a = b = x;
  asm("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 0" : "+v"(a), "+v"(b));
}
DEVINLINE void sr_both32(float x, float& a, float& b) {
  a = b = x;
  asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 0" : "+v"(a), "+v"(b));
}
template <class F>
DEVINLINE float sr_reduce(float x, F f) {
  x = f(x, sr_lane<0xb1>(x, x));    // lane ^ 1
  x = f(x, sr_lane<0x4e>(x, x));    // lane ^ 2
  x = f(x, sr_lane<0x141>(x, x));   // of 8, from the other end
  x = f(x, sr_lane<0x140>(x, x));   // of 16, from the other end
  float a, b;
  sr_both16(x, a, b);
  sr_both32(f(a, b), a, b);
  return f(a, b);
}
DEVINLINE float sr_sum(float x) {
  return sr_reduce(x, [](float a, float b) { return a + b; });
}
DEVINLINE float sr_max(float x) {
  return sr_reduce(x, [](float a, float b) { return fmaxf(a, b); });
}
template <class T>
DEVINLINE T sr_scan(T x) {
  x += sr_lane<0x111>(x, T(0));        // the lane 1, 2, 4, 8 below in its 16
  x += sr_lane<0x112>(x, T(0));
  x += sr_lane<0x114>(x, T(0));
  x += sr_lane<0x118>(x, T(0));
  x += sr_lane<0x142, 0xa>(x, T(0));   // the last of the 16 below
  x += sr_lane<0x143, 0xc>(x, T(0));   // the last of the lower half
  return x;
}

// Constants that unpack a dword of two bf16.  Every pass asks for its own,
// which the compiler cannot see to be the same: it would otherwise keep one
// pass's unpacked row for the next, twice the registers there are.
struct Unpack {
  uint32_t shift = 16, high = 0xffff0000u, sign = 0x000f000fu;
  DEVINLINE Unpack() {
    asm volatile("" : "+s"(shift), "+s"(high), "+s"(sign));
  }
  DEVINLINE float lo(uint32_t u) const {
    return __builtin_bit_cast(float, u << shift);
  }
  DEVINLINE float hi(uint32_t u) const {
    return __builtin_bit_cast(float, u & high);
  }
  // both halves as monotone keys (bf16_key)
  DEVINLINE uint32_t keys(uint32_t u) const {
    typedef __attribute__((ext_vector_type(2))) short short2v;
    const short2v neg =
        __builtin_bit_cast(short2v, u) >> __builtin_bit_cast(short2v, sign);
    return u ^ (__builtin_bit_cast(uint32_t, neg) | 0x80008000u);
  }
  // and back
  DEVINLINE uint32_t bits(uint32_t k) const {
    typedef __attribute__((ext_vector_type(2))) short short2v;
    const short2v pos =
        __builtin_bit_cast(short2v, k) >> __builtin_bit_cast(short2v, sign);
    return k ^ (~__builtin_bit_cast(uint32_t, pos) | 0x80008000u);
  }
  // the halves of a pair of keys
  DEVINLINE uint32_t first(uint32_t k) const { return k & ~high; }
  DEVINLINE uint32_t second(uint32_t k) const { return k >> shift; }
};

// Largest of eight keys.  Written out so that a pass computes its own: the
// compiler would keep all of them over the loop of the windows.
DEVINLINE uint32_t largest_key(const uint32_t (&k)[4]) {
  uint32_t m;
  asm volatile(
      "v_pk_max_u16 %0, %1, %2\n\tv_pk_max_u16 %0, %0, %3\n\t"
      "v_pk_max_u16 %0, %0, %4"
      : "=&v"(m)
      : "v"(k[0]), "v"(k[1]), "v"(k[2]), "v"(k[3]));
  return max(m & 0xffffu, m >> 16);
}

// Whether any of eight keys is one of two (each given twice in a dword).
DEVINLINE bool has_key(const uint32_t (&k)[4], const uint32_t (&same)[2]) {
  typedef __attribute__((ext_vector_type(2))) unsigned short ushort2v;
  ushort2v m = {0xffff, 0xffff};
#pragma unroll
  for (int q = 0; q < 4; ++q)
#pragma unroll
    for (int i = 0; i < 2; ++i)
      m = __builtin_elementwise_min(m,
                                    __builtin_bit_cast(ushort2v, k[q] ^ same[i]));
  return m.x == 0 || m.y == 0;
}

DEVINLINE float bf16_key_val(uint32_t key) {
  const uint32_t u = (key & 0x8000u) ? key ^ 0x8000u : key ^ 0xffffu;
  return bf16_val((uint16_t)u);
}

template <int NCH>
__global__
__launch_bounds__(SR_THREADS, NCH > 8 ? 2 : 4) void sample_bf16_resident_kernel(
    int32_t* __restrict__ out,             // [B]
    const uint16_t* __restrict__ logits,   // [B, V] bf16 bits
    const float* __restrict__ temperature, // [B]
    const int32_t* __restrict__ top_k,     // [B] (<=0 => disabled)
    const float* __restrict__ top_p,       // [B] (>=1 => disabled)
    const float* __restrict__ uniforms,    // [B]
    int V) {
  __shared__ float red[SR_WAVES];
  __shared__ uint32_t bins[SR_WINDOW + WAVE_SIZE];
  __shared__ uint4 list_k[SR_LIST];    // chunks of the first window: keys
  __shared__ int list_at[SR_LIST];     // and number
  __shared__ __attribute__((aligned(16))) int kept_at[SR_THREADS];
  __shared__ float kept_w[SR_THREADS], sorted_w[SR_THREADS];
  __shared__ int kept_e[SR_THREADS], sorted_e[SR_THREADS];
  __shared__ int s_list, s_kept, s_last;
  __shared__ uint32_t wave_n[SR_WAVES];
  __shared__ float wave_w[SR_WAVES];
  __shared__ int s_tau, s_top, s_cell;
  __shared__ float s_base;
  __shared__ uint32_t s_pick;
  __shared__ float cells[NCH * SR_WAVES];

  const int seq = blockIdx.x;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const uint16_t* row = logits + (int64_t)seq * V;
  const float temp = temperature[seq];
  const bool greedy = temp <= 0.0f;
  const float inv_t = greedy ? 1.0f : 1.0f / temp;

  // Element h of chunk j is logit (j * 512 + tid) * 8 + h; past the end -inf.
  // The chunk that the row ends in is loaded once, for whichever it is: with a
  // check in all of them the code of the loads alone was a third of the kernel,
  // which then did not fit the instruction cache.
  constexpr int CHUNK = SR_THREADS * 8;
  const int whole = V / CHUNK;
  uint32_t d[NCH][4];
#pragma unroll
  for (int j = 0; j < NCH; ++j) {
    if (j < whole) {
      typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
      const u32x4 v = __builtin_nontemporal_load(
          reinterpret_cast<const u32x4*>(row + (j * SR_THREADS + tid) * 8));
      d[j][0] = v.x; d[j][1] = v.y; d[j][2] = v.z; d[j][3] = v.w;
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) d[j][q] = 0xff80ff80u;
    }
  }
  if (whole * CHUNK < V) {
    const int at = (whole * SR_THREADS + tid) * 8;
    uint32_t end[4];
    if (at + 8 <= V) {
      const uint4 v = *reinterpret_cast<const uint4*>(row + at);
      end[0] = v.x; end[1] = v.y; end[2] = v.z; end[3] = v.w;
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int e = at + 2 * q;
        const uint32_t lo = e < V ? row[e] : 0xff80u;
        const uint32_t hi = e + 1 < V ? row[e + 1] : 0xff80u;
        end[q] = lo | (hi << 16);
      }
    }
#pragma unroll
    for (int j = 0; j < NCH; ++j)
      if (j == whole) {
#pragma unroll
        for (int q = 0; q < 4; ++q) d[j][q] = end[q];
      }
  }
  // ---- maximum ----
  float mx = -INFINITY;
  {
    const Unpack un;
#pragma unroll
    for (int j = 0; j < NCH; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        mx = fmaxf(fmaxf(mx, un.lo(d[j][q])), un.hi(d[j][q]));
  }
  mx = sr_max(mx);
  if (lane == 0) red[wave] = mx;
  if (tid == 0) s_pick = 0xffffffffu;
  __syncthreads();
  float M = red[0];
#pragma unroll
  for (int w = 1; w < SR_WAVES; ++w) M = fmaxf(M, red[w]);

  const int k = top_k[seq];
  const float p = top_p[seq];
  const bool do_k = k > 0 && k < V;
  const bool do_p = p < 1.0f && !greedy;
  const float rate = inv_t * 1.44269504088896340736f;   // to powers of two
  auto weight = [&](float x) {
    return __builtin_amdgcn_exp2f((x - M) * rate);
  };

  float target_p = 0.0f;
  if (do_p) {
    const Unpack un;
    float z = 0.0f;
#pragma unroll
    for (int j = 0; j < NCH; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        z += weight(un.lo(d[j][q])) + weight(un.hi(d[j][q]));
    z = sr_sum(z);
    __syncthreads();  // red was read by everybody
    if (lane == 0) red[wave] = z;
    __syncthreads();
    z = 0.0f;
#pragma unroll
    for (int w = 0; w < SR_WAVES; ++w) z += red[w];
    target_p = p * z;
  }

  // From here on the row is kept as keys: a chunk's largest takes a few
  // instructions, and a wave passes over the chunks of which none matters.
  {
    const Unpack un;
#pragma unroll
    for (int j = 0; j < NCH; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) d[j][q] = un.keys(d[j][q]);
  }
  int max_key = 0x8000;  // key of the maximum (of +0 for either zero)
  if (M != 0.0f)
    max_key =
        (int)bf16_key((uint16_t)(__builtin_bit_cast(uint32_t, M) >> 16));
  // Lowest index of the maximum (all threads call it); -0 is as large as +0.
  auto first_max = [&]() {
    const uint32_t low = M == 0.0f ? 0x7fffu : (uint32_t)max_key;
    const uint32_t same[2] = {(uint32_t)max_key * 0x10001u, low * 0x10001u};
    uint32_t at = 0, e[4] = {0, 0, 0, 0};
    bool any = false;
#pragma unroll
    for (int j = NCH - 1; j >= 0; --j)
      if (largest_key(d[j]) >= low && has_key(d[j], same)) {
        any = true;
        at = (j * SR_THREADS + tid) * 8;
#pragma unroll
        for (int q = 0; q < 4; ++q) e[q] = d[j][q];
      }
    if (any) {
      uint32_t first = 8;
#pragma unroll
      for (int h = 7; h >= 0; --h) {
        const uint32_t key = (h & 1) ? e[h >> 1] >> 16 : e[h >> 1] & 0xffffu;
        if (key == low || key == (uint32_t)max_key) first = h;
      }
      atomicMin(&s_pick, at + first);
    }
    __syncthreads();
    if (tid == 0)   // what is past the end is no logit
      out[seq] = M == -INFINITY && !greedy ? 0
                 : s_pick < (uint32_t)V    ? (int32_t)s_pick
                                           : -1;
  };
  if (greedy) {
    first_max();
    return;
  }

  // ---- thresholds ----
  int tau = 0;
  int listed = -1;   // chunks in the list, when that is all that is kept
  if (do_k || do_p) {
    int top = max_key;
    // The chunks with a key of the first window go to a list in LDS: they are
    // few, and what is done with them is a loop and not the code of NCH chunks.
    if constexpr (NCH > 8) {
      if (tid == 0) s_list = 0;
      __syncthreads();
      const uint32_t low = (uint32_t)max(top - SR_FIRST + 1, 0);
#pragma unroll
      for (int j = 0; j < NCH; ++j)
        if (largest_key(d[j]) >= low) {
          const int at = atomicAdd(&s_list, 1);
          if (at < SR_LIST) {
            list_k[at] = make_uint4(d[j][0], d[j][1], d[j][2], d[j][3]);
            list_at[at] = j * SR_THREADS + tid;
          }
        }
      __syncthreads();
      if (s_list <= SR_LIST) listed = s_list;
    }
    uint32_t seen_n = 0;   // above the window
    float seen_w = 0.0f;
    int width = SR_FIRST;
    while (true) {
      for (int b = tid; b < width; b += SR_THREADS) bins[b] = 0;
      if (tid == 0) {
        s_tau = -1;
        s_top = -1;
      }
      __syncthreads();
      // an element outside the window counts where nobody looks
      const uint32_t spare = (uint32_t)(SR_WINDOW + lane);
      auto count = [&](uint32_t k0, uint32_t k1) {
        const uint32_t b0 = (uint32_t)top - k0, b1 = (uint32_t)top - k1;
        atomicAdd(&bins[b0 < (uint32_t)width ? b0 : spare], 1u);
        atomicAdd(&bins[b1 < (uint32_t)width ? b1 : spare], 1u);
      };
      if (NCH > 8 && width == SR_FIRST && listed >= 0) {
        const uint32_t* list = reinterpret_cast<const uint32_t*>(list_k);
        for (int e = tid; e < listed * 4; e += SR_THREADS)
          count(list[e] & 0xffffu, list[e] >> 16);
      } else {
        const Unpack un;
        const uint32_t low = (uint32_t)max(top - width + 1, 0);
#pragma unroll
        for (int j = 0; j < NCH; ++j)
          if (largest_key(d[j]) >= low) {
#pragma unroll
            for (int q = 0; q < 4; ++q)
              count(un.first(d[j][q]), un.second(d[j][q]));
          }
      }
      __syncthreads();
      // thread t takes the keys top - (per t + i), i < per, in order
      const int per = width / SR_THREADS > 0 ? width / SR_THREADS : 1;
      const bool has = tid * per < width;
      uint32_t n = 0;
      float w = 0.0f;
      if (has)
        for (int i = 0; i < per; ++i) {
          const int b = tid * per + i;
          const uint32_t c = bins[b];
          if (c) {
            n += c;
            w += (float)c * weight(bf16_key_val((uint32_t)(top - b)));
          }
        }
      // inclusive sums over the wave, then over the waves before it
      const uint32_t sn = sr_scan(n);
      const float sw = sr_scan(w);
      if (lane == 63) {
        wave_n[wave] = sn;
        wave_w[wave] = sw;
      }
      __syncthreads();
      uint32_t all_n = seen_n, base_n = 0;
      float all_w = seen_w, base_w = 0.0f;
#pragma unroll
      for (int v = 0; v < SR_WAVES; ++v) {
        if (v == wave) {
          base_n = all_n;
          base_w = all_w;
        }
        all_n += wave_n[v];
        all_w += wave_w[v];
      }
      if (has) {
        uint32_t cn = base_n + sn - n;
        float cw = base_w + sw - w;
        const bool end_k = do_k && cn + n >= (uint32_t)k;
        const bool end_p = do_p && base_w + sw >= target_p;
        if (n && (end_k || end_p)) {
          // the first key, from the top, at which either is reached; the sums
          // in this order may end a rounding step below the scanned ones: then
          // the last key with a logit
          int reached = -1;
          for (int i = 0; i < per; ++i) {
            const int b = tid * per + i;
            const uint32_t c = bins[b];
            if (!c) continue;
            cn += c;
            cw += (float)c * weight(bf16_key_val((uint32_t)(top - b)));
            reached = top - b;
            if ((do_k && cn >= (uint32_t)k) || (do_p && cw >= target_p)) break;
          }
          atomicMax(&s_tau, reached);
        }
      }
      __syncthreads();
      tau = s_tau;
      if (tau >= 0) break;
      if (width == SR_FIRST) {   // the second window follows the first
        top -= SR_FIRST;
      } else {
        // the highest key below the window
        const int lo = top - width + 1;
        int next = -1;
        const Unpack un;
#pragma unroll
        for (int j = 0; j < NCH; ++j)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const int k0 = (int)un.first(d[j][q]);
            const int k1 = (int)un.second(d[j][q]);
            if (k0 < lo) next = max(next, k0);
            if (k1 < lo) next = max(next, k1);
          }
        if (next >= 0) atomicMax(&s_top, next);
        __syncthreads();
        top = s_top;
      }
      listed = -1;
      seen_n = all_n;
      seen_w = all_w;
      width = width < SR_SECOND ? SR_SECOND : SR_WINDOW;
      if (top < 0) {  // everything is kept (p * Z not reached by rounding)
        tau = 0;
        break;
      }
      __syncthreads();  // s_top and the bins are reset above
    }
  }

  const uint32_t utau = (uint32_t)tau;
  auto kept = [&](uint32_t key) {
    return key >= utau ? weight(bf16_key_val(key)) : 0.0f;
  };
  auto kept_sum = [&](const uint32_t* e) {
    float sum = 0.0f;
    for (int q = 0; q < 4; ++q) sum += kept(e[q] & 0xffffu) + kept(e[q] >> 16);
    return sum;
  };
  // the element of a chunk at which the running sum passes, or the last with
  // mass
  auto element = [&](const uint32_t* e, float run, float target) {
    int chosen = 0;
    for (int h = 0; h < 8; ++h) {
      const float w = kept((h & 1) ? e[h >> 1] >> 16 : e[h >> 1] & 0xffffu);
      run += w;
      if (w > 0.0f) chosen = h;
      if (w > 0.0f && run > target) break;
    }
    return chosen;
  };

  // ---- listed: at most as many kept chunks as threads are put in order ----
  if (NCH > 8 && listed >= 0) {
    if (tid == 0) {
      s_kept = 0;
      s_cell = INT_MAX;
      s_last = -1;
    }
    __syncthreads();
    for (int e = tid; e < listed; e += SR_THREADS) {
      const uint32_t* k = reinterpret_cast<const uint32_t*>(list_k + e);
      uint32_t most = 0;
      for (int q = 0; q < 4; ++q) most = max(most, max(k[q] & 0xffffu, k[q] >> 16));
      if (most >= utau) {
        const int at = atomicAdd(&s_kept, 1);
        if (at < SR_THREADS) {
          kept_at[at] = list_at[e];
          kept_w[at] = kept_sum(k);
          kept_e[at] = e;
        }
      }
    }
    __syncthreads();
    const int n = s_kept;
    if (n <= SR_THREADS) {
      if (tid >= n) kept_at[tid] = INT_MAX;
      __syncthreads();
      if (tid < n) {
        const int own = kept_at[tid];
        int rank = 0;
        for (int e = 0; e < n; e += 4) {
          const int4 v = *reinterpret_cast<const int4*>(kept_at + e);
          rank += (v.x < own) + (v.y < own) + (v.z < own) + (v.w < own);
        }
        sorted_w[rank] = kept_w[tid];
        sorted_e[rank] = kept_e[tid];
      }
      __syncthreads();
      const float w = tid < n ? sorted_w[tid] : 0.0f;
      const float own = sr_scan(w);
      if (lane == 63) wave_w[wave] = own;
      __syncthreads();
      float before = 0.0f, total = 0.0f;
#pragma unroll
      for (int v = 0; v < SR_WAVES; ++v) {
        if (v == wave) before = total;
        total += wave_w[v];
      }
      if (total > 0.0f) {
        const float target = uniforms[seq] * total;
        if (w > 0.0f) {
          if (before + own > target) atomicMin(&s_cell, tid);
          atomicMax(&s_last, tid);
        }
        __syncthreads();
        const bool passed = s_cell != INT_MAX;
        if (tid == (passed ? s_cell : s_last)) {
          const int e = sorted_e[tid];
          out[seq] = list_at[e] * 8 +
                     element(reinterpret_cast<const uint32_t*>(list_k + e),
                             before + own - w, passed ? target : INFINITY);
        }
      } else {   // as below
        first_max();
      }
      return;
    }
    __syncthreads();   // s_cell is used again
  }

  // ---- kept mass of every (chunk, wave), in index order ----
  const Unpack un;
#pragma unroll
  for (int j = 0; j < NCH; ++j) {
    float sum = 0.0f;
    if (__any(largest_key(d[j]) >= utau)) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const uint32_t v = un.bits(d[j][q]);
        const float w0 = weight(un.lo(v)), w1 = weight(un.hi(v));
        sum += (un.first(d[j][q]) >= utau ? w0 : 0.0f) +
               (un.second(d[j][q]) >= utau ? w1 : 0.0f);
      }
      sum = sr_sum(sum);
    }
    if (lane == 0) cells[j * SR_WAVES + wave] = sum;
  }
  __syncthreads();
  // wave 0: the first cell whose running sum passes u * total
  if (wave == 0) {
    constexpr int PER = (NCH * SR_WAVES + 63) / 64;
    float own = 0.0f;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int c = lane * PER + i;
      own += c < NCH * SR_WAVES ? cells[c] : 0.0f;
    }
    float run = sr_scan(own);
    const float total = __shfl(run, 63, 64);
    const float target = uniforms[seq] * total;
    run -= own;
    int cell = -1;       // first that passes the target
    int last = -1;       // last with any mass
    float base = 0.0f;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int c = lane * PER + i;
      const float w = c < NCH * SR_WAVES ? cells[c] : 0.0f;
      if (w > 0.0f) last = c;
      if (cell < 0 && w > 0.0f && run + w > target) {
        cell = c;
        base = run;
      }
      run += w;
    }
    const uint64_t found = __ballot(cell >= 0), any = __ballot(last >= 0);
    float rest = INFINITY;   // mass into the cell; infinite: its last element
    int pick = -1;
    if (!(total > 0.0f)) {
      // nothing that could be drawn from: the largest logit
    } else if (found) {
      const int l = __builtin_ctzll(found);
      pick = __shfl(cell, l, 64);
      rest = target - __shfl(base, l, 64);
    } else if (any) {
      pick = __shfl(last, 63 - __builtin_clzll(any), 64);
    }
    if (lane == 0) {
      s_cell = pick;
      s_base = rest;
    }
  }
  __syncthreads();
  const int cell = s_cell;
  if (cell < 0) {
    // A kept logit that is not a number, or an infinite one, leaves no mass
    // to draw from: the largest logit, the first one where none is above
    // minus infinity.
    first_max();
    return;
  }
  if (wave == cell % SR_WAVES) {
    uint32_t e[4] = {0, 0, 0, 0};
#pragma unroll
    for (int j = 0; j < NCH; ++j)
      if (j == cell / SR_WAVES) {
#pragma unroll
        for (int q = 0; q < 4; ++q) e[q] = d[j][q];
      }
    const float sum = kept_sum(e);
    const float run = sr_scan(sum);
    const float rest = s_base;
    const uint64_t past = __ballot(sum > 0.0f && run > rest);
    const uint64_t some = __ballot(sum > 0.0f);
    const int l = past ? __builtin_ctzll(past) : 63 - __builtin_clzll(some);
    if (lane == l)
      out[seq] = ((cell / SR_WAVES) * SR_THREADS + tid) * 8 +
                 element(e, run - sum, rest);
  }
}

// ---------------------------------------------------------------------------
// bf16 rows of more than 65536 logits (up to 262144): one pass over the row, a
// wave at a time 2048 logits that lie together (a unit), the next unit's loads under
// way, so that rows of several workgroups and their arithmetic overlap.  The pass
// leaves
//
//   * the largest logit of every lane;
//   * where top-p or no limit needs them, the mass of every unit, each with its own
//     largest as reference (scaled to the row's maximum afterwards: one rounding);
//   * a list of the chunks of eight that can hold a kept logit.  With top-k these
//     are the ones at or above a bound: every wave knows the ceil(k / waves)-th of
//     its lanes' maxima, at least k logits are at or above the least of those.
//     With top-p alone: an octave below the largest so far, where the logits of the
//     first step that are listed hold p of that step's mass;
//   * otherwise (a flat top-p, a k of more than 32 a wave) the counts of all keys in
//     a window around the first step's maximum.
//
// Thresholds come from the counts as in the resident kernel; those of a short
// list every wave finds for itself, and up to 64 kept chunks one wave puts in order.
// A row without limits is drawn from the units' masses, of which one is read
// again; so is a row whose list does not hold all that is kept, by another pass for
// the kept masses.  Whatever else can be met (a threshold below the window, a
// sum that is not a number) is done by further passes over memory from the top
// key down: rare, and written as loops.
//
// Bound: HBM with greedy rows (1024 of 128256: 41.6 us, 6.3 TB/s) and with sampled
// ones without limits (50 us); an exponential is four cycles a logit of the 7 us a
// row's arithmetic takes; then the serial end of a row, four barriers.
// 1024 rows of 128256, greedy / top-k 50 and top-p / top-p 0.9 / top-k 40 / no limits /
// mixed: 41.6, 62, 124, 54, 50 and 77 us; held in registers, one row a compute unit
// whose passes follow its loads, 54, 123, 185, 99, 103 and 140.  64 rows mixed 39.9 for
// 42.5.  A flat top-p row takes twice as long as another: of more rows than are on
// the chip at once (two a compute unit) those start first, which costs a
// microsecond a row (1024 mixed rows in the order of the call 92 us, so 77); so do
// rows of a top-k that no list serves (a tenth of k = 500 among others of top-k 50 and
// top-p, 600 / 1024 / 2000 rows 69.9 90.6 154, so 51.4 76.5 134).  Up to 65536 logits the register kernel has
// two rows on a unit and is ahead (1024 of 49000, mixed, 49.3, here 50.7; of 32000 36.3
// and 43).  Just beyond, held in registers and here, 256 rows of 65544: top-k 50 and
// top-p 26.9 and 18.9, top-k 40 22.1 and 16.8, no limits 20.5 and 14.0, greedy 10.9 and
// 10.1, mixed 31.0 and 31.1, but rows that are read again are behind there, top-p 0.9
// 31.7 and 33.8, k = 500 27.5 and 29.8 (64 rows 29.9 29.8 and 25.7 27.6; 300 rows 57.4
// 41.0 and 48.3 35.5; 256 rows of 128256 53.3 47.8 and 41.4 36.8, one of k = 500 27.0 and
// 29.8).  That second read is not it: plain loads in the first pass of such rows, for
// the caches to keep them, change nothing at any of these sizes.
//
// Thresholds, ordered draw and `element` repeat the resident kernel's on another
// list: what is mended in one is looked for in the other.
// ---------------------------------------------------------------------------
constexpr int SS_U = 4;                  // chunks of eight a lane in a unit
constexpr int SS_UNIT = SS_U * 512;      // logits
constexpr int SS_UNITS = 128;            // of a row at most
constexpr int SS_WINDOW = 4096;          // keys that are counted at a time
constexpr int SS_OCTAVE = 128;           // keys of an octave
constexpr int SS_ABOVE = 512;            // of the window, above the first maximum
constexpr int SS_NARROW = 512;           // keys that a wave looks through alone
constexpr int SS_ORDERED = 4096;         // rows that are put in order: 64 words

// Not fmaxf, which would quiet each operand first; rows with a NaN are found by
// their bits or their mass and done again.
DEVINLINE float ss_max3(float a, float b, float c) {
  float m;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(m) : "v"(a), "v"(b), "v"(c));
  return m;
}
DEVINLINE uint32_t ss_pk_max(uint32_t a, uint32_t b) {
  uint32_t m;
  asm("v_pk_max_u16 %0, %1, %2" : "=v"(m) : "v"(a), "v"(b));
  return m;
}

// Two bins of a window of SS_WINDOW keys from `top` down, `spare` outside of it.
DEVINLINE uint32_t ss_bins(uint32_t keys, uint32_t top, uint32_t spare) {
  typedef __attribute__((ext_vector_type(2))) unsigned short ushort2v;
  const ushort2v b = __builtin_bit_cast(ushort2v, top) -
                     __builtin_bit_cast(ushort2v, keys);
  return __builtin_bit_cast(
      uint32_t,
      __builtin_elementwise_min(b, __builtin_bit_cast(ushort2v, spare)));
}

// Row of a workgroup when those that can take another pass (a top-k that no list
// serves, top-p without a top-k) start first.  Every wave finds it for itself from
// the rows' settings, 64 rows in a word of `words`, which is free again behind the
// next barrier.
template <int WAVES>
DEVINLINE int ss_long_first(uint64_t* words, int wave, int V,
                            const float* temperature, const int32_t* top_k,
                            const float* top_p) {
  const int lane = threadIdx.x & 63, B = gridDim.x;
  const int groups = (B + 63) / 64;
  for (int g = wave; g < groups; g += WAVES) {
    const int r = min(g * 64 + lane, B - 1);
    const int k = top_k[r];
    const bool later =
        temperature[r] <= 0.0f ||
        (k > 0 && k < V ? k <= 32 * WAVES : !(top_p[r] < 1.0f));
    const uint64_t word = __ballot(!later && g * 64 + lane < B);
    if (lane == 0) words[g] = word;
  }
  __syncthreads();
  uint64_t own = lane < groups ? words[lane] : 0;
  const int first = __builtin_amdgcn_readlane(sr_scan(__popcll(own)), 63);
  int at = blockIdx.x;
  if (at >= first) {   // among the others
    at -= first;
    const int n = min(max(B - lane * 64, 0), 64);
    own = ~own & (n == 64 ? ~0ull : (1ull << n) - 1);
  }
  const int n = __popcll(own), to = sr_scan(n);
  const int g = __builtin_ctzll(__ballot(to > at));
  at -= __builtin_amdgcn_readlane(to - n, g);
  const uint64_t word =
      (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(own >> 32), g) << 32 |
      (uint32_t)__builtin_amdgcn_readlane((int)own, g);
  const bool mine = (word >> lane & 1) &&
                    __popcll(word & ((1ull << lane) - 1)) == at;
  return g * 64 + __builtin_ctzll(__ballot(mine));
}

template <int SS_THREADS>
__global__ __launch_bounds__(SS_THREADS, 4) void sample_bf16_stream_kernel(
    int32_t* __restrict__ out,             // [B]
    const uint16_t* __restrict__ logits,   // [B, V] bf16 bits
    const float* __restrict__ temperature, // [B]
    const int32_t* __restrict__ top_k,     // [B] (<=0 => disabled)
    const float* __restrict__ top_p,       // [B] (>=1 => disabled)
    const float* __restrict__ uniforms,    // [B]
    int V, bool ordered) {
  constexpr int SS_WAVES = SS_THREADS / WAVE_SIZE;
  constexpr int SS_LIST = SS_THREADS == 512 ? 3072 : 4096;   // as the LDS takes
  constexpr int U = SS_U, UNIT = SS_UNIT;
  __shared__ __attribute__((aligned(16))) uint32_t
      bins[SS_WINDOW + WAVE_SIZE > 4 * SS_THREADS ? SS_WINDOW + WAVE_SIZE
                                                 : 4 * SS_THREADS];
  __shared__ __attribute__((aligned(16))) int kept_at[SS_THREADS];
  __shared__ uint4 list_k[SS_LIST];    // listed chunks: logits
  __shared__ int list_at[SS_LIST];     // and number
  // behind the counts, where they were
  int* const kept_e = reinterpret_cast<int*>(bins);
  int* const sorted_e = kept_e + SS_THREADS;
  float* const kept_w = reinterpret_cast<float*>(sorted_e + SS_THREADS);
  float* const sorted_w = kept_w + SS_THREADS;
  // cells: before them the words of ss_long_first
  __shared__ __attribute__((aligned(16))) float cells[SS_UNITS], cell_c[SS_UNITS];
  __shared__ float red[SS_WAVES];
  __shared__ uint32_t bound[SS_WAVES], bound0[SS_WAVES];
  __shared__ uint32_t wave_n[SS_WAVES];
  __shared__ float wave_w[SS_WAVES];
  __shared__ int s_list, s_bad, s_kept, s_last, s_tau, s_top, s_cell;
  __shared__ uint32_t s_pick;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int seq =
      ordered ? ss_long_first<SS_WAVES>(reinterpret_cast<uint64_t*>(cells), wave,
                                        V, temperature, top_k, top_p)
              : blockIdx.x;
  const uint16_t* row = logits + (int64_t)seq * V;
  const float temp = temperature[seq];
  const bool greedy = temp <= 0.0f;
  const float inv_t = greedy ? 1.0f : 1.0f / temp;
  const float rate = inv_t * 1.44269504088896340736f;   // to powers of two
  const int k = top_k[seq];
  const float p = top_p[seq];
  const bool do_k = k > 0 && k < V && !greedy;
  const bool do_p = p < 1.0f && !greedy;
  const bool do_z = !greedy && (do_p || !do_k);   // exponentials of all
  const bool do_list = do_k || do_p;
  const int units = (V + UNIT - 1) / UNIT;

  typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
  // chunk of eight logits at `at`, past the end -inf
  auto load_chunk = [&](int at, uint32_t (&d)[4]) {
    if (at + 8 <= V) {
      const u32x4 v =
          __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(row + at));
      d[0] = v.x; d[1] = v.y; d[2] = v.z; d[3] = v.w;
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int e = at + 2 * q;
        const uint32_t lo = e < V ? row[e] : 0xff80u;
        const uint32_t hi = e + 1 < V ? row[e + 1] : 0xff80u;
        d[q] = lo | (hi << 16);
      }
    }
  };
  auto load = [&](int unit, uint32_t (&d)[U][4]) {
    const int at = unit * UNIT + lane * 8;
    if ((unit + 1) * UNIT <= V) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const u32x4* from = reinterpret_cast<const u32x4*>(row + at + u * 512);
        const u32x4 v = __builtin_nontemporal_load(from);
        d[u][0] = v.x; d[u][1] = v.y; d[u][2] = v.z; d[u][3] = v.w;
      }
    } else {
#pragma unroll
      for (int u = 0; u < U; ++u) load_chunk(at + u * 512, d[u]);
    }
  };
  // f(unit, logits) of this wave's units, the next one's loads under way
  auto for_units = [&](auto&& f) {
    uint32_t d[U][4], e[U][4];
    int unit = wave;
    if (unit < units) load(unit, d);
    while (unit < units) {
      if (unit + SS_WAVES < units) load(unit + SS_WAVES, e);
      f(unit, d);
      unit += SS_WAVES;
      if (unit >= units) break;
      if (unit + SS_WAVES < units) load(unit + SS_WAVES, d);
      f(unit, e);
      unit += SS_WAVES;
    }
  };

  // ---- the row, once: largest, mass, list ----
  const int active = min(SS_WAVES, units);
  // lanes of a wave at or above its bound; of its largest, if that is wanted
  const int share = do_k ? (k + active - 1) / active : 1;
  const bool octave = !do_k || share > 32;
  const int need = octave ? 1 : share;
  float best = -INFINITY;   // of this lane
  int best_at = 0;          // the unit it came with
  uint32_t odd = 0;         // largest bits without the sign, both halves
  int anchor = -1;          // key of the first bin, where all are counted
  if (do_list) {
    for (int b = tid; b < SS_WINDOW; b += SS_THREADS) bins[b] = 0;
    kept_at[tid] = INT_MAX;
  }
  if (tid == 0) {
    s_list = 0;
    s_bad = 0;
    s_kept = 0;
    s_tau = -1;
    s_top = -1;
    s_cell = INT_MAX;
    s_last = -1;
    s_pick = 0xffffffffu;
  }
  const float u01 = uniforms[seq];
  auto take = [&](int unit, const uint32_t (&d)[U][4], bool first) {
    float most[U];
    const Unpack un;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const float a = ss_max3(un.lo(d[u][0]), un.hi(d[u][0]), un.lo(d[u][1]));
      const float b = ss_max3(un.hi(d[u][1]), un.lo(d[u][2]), un.hi(d[u][2]));
      most[u] = ss_max3(ss_max3(un.lo(d[u][3]), un.hi(d[u][3]), a), b, b);
    }
    float all = most[0];
#pragma unroll
    for (int u = 1; u < U; ++u) all = ss_max3(all, most[u], most[u]);
    if (all > best) {
      best = all;
      best_at = unit;
    }
    if (do_z) {
      const float ref = sr_max(all);
      const float c = ref == -INFINITY ? 0.0f : -(ref * rate);
      float z0 = 0.0f, z1 = 0.0f;
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          z0 += __builtin_amdgcn_exp2f(fmaf(un.lo(d[u][q]), rate, c));
          z1 += __builtin_amdgcn_exp2f(fmaf(un.hi(d[u][q]), rate, c));
        }
      const float z = sr_sum(z0 + z1);
      if (lane == 0 && unit < units) {
        cells[unit] = z;
        cell_c[unit] = c;
      }
    } else {
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int q = 0; q < 4; ++q) odd = ss_pk_max(odd, d[u][q] & 0x7fff7fffu);
    }
    if (do_list) {
      const uint32_t own =
          bf16_key((uint16_t)(__builtin_bit_cast(uint32_t, best) >> 16));
      const int step = unit / SS_WAVES;
      if ((step & (step + 1)) == 0) {   // the bound rises with the logarithm
        uint32_t t = 0;
#pragma unroll
        for (int bit = 15; bit >= 0; --bit) {
          const uint32_t c = t | (1u << bit);
          if (__popcll(__ballot(own >= c)) >= need) t = c;
        }
        if (lane == 0) {
          if (first) bound0[wave] = t;
          __hip_atomic_store(&bound[wave], t, __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_WORKGROUP);
        }
      }
      if (first) {
        __syncthreads();
        if (octave) {
          int top = 0;
          for (int w = 0; w < active; ++w) top = max(top, (int)bound0[w]);
          bool flat = do_k;
          if (!do_k) {
            // mass of what would be listed, and of all, of the logits so far
            const float m = bf16_key_val(max(top, 0x007f));
            const float from = bf16_key_val(max(top - SS_OCTAVE + 1, 0x007f));
            const float c = -(m * rate);
            float above = 0.0f;
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
              for (int q = 0; q < 4; ++q) {
                const float lo = un.lo(d[u][q]), hi = un.hi(d[u][q]);
                const float w0 = __builtin_amdgcn_exp2f(fmaf(lo, rate, c));
                const float w1 = __builtin_amdgcn_exp2f(fmaf(hi, rate, c));
                above += (lo >= from ? w0 : 0.0f) + (hi >= from ? w1 : 0.0f);
              }
            above = sr_sum(above);
            if (lane == 0) wave_w[wave] = above;
            __syncthreads();
            above = sr_sum(lane < active ? wave_w[lane] : 0.0f);
            const float z = sr_sum(
                lane < active && cells[lane] > 0.0f
                    ? cells[lane] * __builtin_amdgcn_exp2f(
                                        fmaf(-m, rate, -cell_c[lane]))
                    : 0.0f);
            flat = !(above >= p * z);
          }
          if (flat) anchor = min(top + SS_ABOVE, 0xff80);
        }
      }
      if (anchor >= 0 && unit < units) {
        const uint32_t top = (uint32_t)anchor * 0x10001u;
        // an element outside the window counts where nobody looks
        const uint32_t spare = (uint32_t)(SS_WINDOW + lane) * 0x10001u;
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const uint32_t b = ss_bins(un.keys(d[u][q]), top, spare);
            atomicAdd(&bins[b & 0xffffu], 1u);
            atomicAdd(&bins[b >> 16], 1u);
          }
      }
      uint32_t low = octave ? 0 : 0xffffffffu;
      for (int w = 0; w < active; ++w) {
        const uint32_t b = __hip_atomic_load(&bound[w], __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_WORKGROUP);
        low = octave ? max(low, b) : min(low, b);
      }
      if (octave) low = (uint32_t)max((int)low - SS_OCTAVE + 1, 0);
      const float from = bf16_key_val(max(low, 0x007fu));
      if (anchor < 0 && unit < units && __any(all >= from)) {
        uint64_t at[U];
        int n = 0;
#pragma unroll
        for (int u = 0; u < U; ++u) {
          at[u] = __ballot(most[u] >= from);
          n += __popcll(at[u]);
        }
        int base = 0;
        if (lane == 0) base = atomicAdd(&s_list, n);
        base = __builtin_amdgcn_readfirstlane(base);
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int to = base + __builtin_amdgcn_mbcnt_hi(
                                    (uint32_t)(at[u] >> 32),
                                    __builtin_amdgcn_mbcnt_lo((uint32_t)at[u], 0));
          if ((at[u] >> lane & 1) && to < SS_LIST) {
            list_k[to] = make_uint4(d[u][0], d[u][1], d[u][2], d[u][3]);
            list_at[to] = unit * (UNIT / 8) + u * 64 + lane;
          }
          base += __popcll(at[u]);
        }
      }
    }
  };
  {
    uint32_t d[U][4], e[U][4];
    int unit = wave;
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int q = 0; q < 4; ++q) d[u][q] = 0xff80ff80u;
    if (unit < units) load(unit, d);
    __syncthreads();   // s_list
    bool first = true;
    while (true) {
      if (unit + SS_WAVES < units) load(unit + SS_WAVES, e);
      take(unit, d, first);
      first = false;
      unit += SS_WAVES;
      if (unit >= units) break;
      if (unit + SS_WAVES < units) load(unit + SS_WAVES, d);
      take(unit, e, false);
      unit += SS_WAVES;
      if (unit >= units) break;
    }
  }
  if (__any((odd & 0xffffu) > 0x7f80u || (odd >> 16) > 0x7f80u) && lane == 0)
    s_bad = 1;
  {
    const float m = sr_max(best);
    if (lane == 0) red[wave] = m;
  }
  __syncthreads();
  float M = red[0];
#pragma unroll
  for (int w = 1; w < SS_WAVES; ++w) M = fmaxf(M, red[w]);
  bool bad = s_bad;

  // Mass of a unit with M's weight 1 (0 stays: its own scale may be infinite).
  auto cell = [&](int c) {
    const float z = c < units ? cells[c] : 0.0f;
    return z > 0.0f
               ? z * __builtin_amdgcn_exp2f(fmaf(-M, rate, -cell_c[c]))
               : z;
  };
  float Z = 0.0f;
  if (do_z) {
#pragma unroll
    for (int i = 0; i < SS_UNITS / 64; ++i) Z += cell(i * 64 + lane);
    Z = sr_sum(Z);
    bad = !(Z > 0.0f && Z < INFINITY);
  }
  bad = bad || M == -INFINITY;

  // Lowest index of the largest logit that is a number (all threads call it).
  auto first_max = [&]() {
    for (int at = tid * 8; at < V; at += SS_THREADS * 8) {
      uint32_t d[4];
      load_chunk(at, d);
      const Unpack un;
      uint32_t h = 8;
#pragma unroll
      for (int q = 3; q >= 0; --q) {
        if (un.hi(d[q]) == M) h = 2 * q + 1;
        if (un.lo(d[q]) == M) h = 2 * q;
      }
      if (h < 8) {
        atomicMin(&s_pick, at + h);
        break;
      }
    }
    __syncthreads();
    if (tid == 0)   // what is past the end is no logit
      out[seq] = M == -INFINITY && !greedy ? 0
                 : s_pick < (uint32_t)V    ? (int32_t)s_pick
                                           : -1;
  };
  if (bad) {   // the maximum of the numbers, by comparisons that pass over others
    float m = -INFINITY;
    for (int at = tid * 8; at < V; at += SS_THREADS * 8) {
      uint32_t d[4];
      load_chunk(at, d);
      const Unpack un;
      for (int q = 0; q < 4; ++q) {
        const float lo = un.lo(d[q]), hi = un.hi(d[q]);
        m = lo > m ? lo : m;
        m = hi > m ? hi : m;
      }
    }
    m = sr_max(m);
    __syncthreads();   // red was read by everybody
    if (lane == 0) red[wave] = m;
    __syncthreads();
    M = red[0];
#pragma unroll
    for (int w = 1; w < SS_WAVES; ++w) M = fmaxf(M, red[w]);
  }
  if (greedy) {
    if (bad) {
      first_max();
      return;
    }
    if (best == M) {
      uint32_t d[U][4];
      load(best_at, d);
      const Unpack un;
      uint32_t h = 0;
#pragma unroll
      for (int u = U - 1; u >= 0; --u)
#pragma unroll
        for (int q = 3; q >= 0; --q) {
          if (un.hi(d[u][q]) == M) h = u * 512 + 2 * q + 1;
          if (un.lo(d[u][q]) == M) h = u * 512 + 2 * q;
        }
      atomicMin(&s_pick, (uint32_t)(best_at * UNIT + lane * 8) + h);
    }
    __syncthreads();
    if (tid == 0) out[seq] = (int32_t)s_pick;
    return;
  }

  auto weight = [&](float x) {
    return __builtin_amdgcn_exp2f((x - M) * rate);
  };
  if (bad && do_p) {
    float z = 0.0f;
    for (int at = tid * 8; at < V; at += SS_THREADS * 8) {
      uint32_t d[4];
      load_chunk(at, d);
      const Unpack un;
      for (int q = 0; q < 4; ++q) z += weight(un.lo(d[q])) + weight(un.hi(d[q]));
    }
    z = sr_sum(z);
    __syncthreads();   // red was read by everybody
    if (lane == 0) red[wave] = z;
    __syncthreads();
    Z = 0.0f;
#pragma unroll
    for (int w = 0; w < SS_WAVES; ++w) Z += red[w];
  }
  const float target_p = p * Z;
  int max_key = 0x8000;  // key of the maximum (of +0 for either zero)
  if (M != 0.0f)
    max_key =
        (int)bf16_key((uint16_t)(__builtin_bit_cast(uint32_t, M) >> 16));

  // ---- thresholds ----
  int tau = 0;
  int listed = -1;   // chunks in the list, when it holds all that is kept
  if (do_list) {
    uint32_t low = octave ? 0 : 0xffffffffu;
    for (int w = 0; w < active; ++w)
      low = octave ? max(low, bound[w]) : min(low, bound[w]);
    if (octave) low = (uint32_t)max((int)low - SS_OCTAVE + 1, 0);
    // whether all from `low` on is listed
    const bool whole = !bad && anchor < 0 && s_list <= SS_LIST;
    int top = max_key, width = SS_WINDOW;
    // whether the bins hold the counts: of all logits, or of the listed ones
    bool counted = false, some = false;
    if (!bad && max_key <= anchor) {
      counted = true;
      top = anchor;
    } else if (whole && top - (int)low < SS_WINDOW) {
      counted = some = true;
      width = max(top - (int)low + 1, 1);
      const Unpack un;
      const uint32_t* list = reinterpret_cast<const uint32_t*>(list_k);
      for (int e = tid; e < s_list * 4; e += SS_THREADS) {
        const uint32_t b =
            ss_bins(un.keys(list[e]), (uint32_t)top * 0x10001u,
                    (uint32_t)(SS_WINDOW + lane) * 0x10001u);
        atomicAdd(&bins[b & 0xffffu], 1u);
        atomicAdd(&bins[b >> 16], 1u);
      }
      __syncthreads();
    }
    if (some && width <= SS_NARROW) {
      // every wave for itself: lane l takes the keys top - (8 l + i), in order
      constexpr int PER = SS_NARROW / 64;
      uint32_t c[PER], n = 0;
      float m[PER], w = 0.0f;
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        const int b = lane * PER + i;
        c[i] = b < width ? bins[b] : 0;
        m[i] = c[i] ? (float)c[i] * weight(bf16_key_val((uint32_t)(top - b)))
                    : 0.0f;
        n += c[i];
        w += m[i];
      }
      const uint32_t sn = sr_scan(n);
      const float sw = sr_scan(w);
      const uint64_t ends = __ballot(n && ((do_k && sn >= (uint32_t)k) ||
                                           (do_p && sw >= target_p)));
      if (ends) {
        // the first key, from the top, at which either is reached; the sums
        // in this order may end a rounding step below the scanned ones: then
        // the last key with a logit
        uint32_t cn = sn - n;
        float cw = sw - w;
        int reached = -1;
        bool done = false;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
          cn += c[i];
          cw += m[i];
          if (c[i] && !done) {
            reached = top - (lane * PER + i);
            done = (do_k && cn >= (uint32_t)k) || (do_p && cw >= target_p);
          }
        }
        tau = __builtin_amdgcn_readlane(reached, __builtin_ctzll(ends));
        listed = s_list;
      } else {
        __syncthreads();   // the bins were read by everybody
        counted = some = false;
        width = SS_WINDOW;
      }
    }
    uint32_t seen_n = 0;   // above the window
    float seen_w = 0.0f;
    while (listed < 0) {
      if (!counted) {
        for (int b = tid; b < width; b += SS_THREADS) bins[b] = 0;
        if (tid == 0) {
          s_tau = -1;
          s_top = -1;
        }
        __syncthreads();
        const uint32_t top2 = (uint32_t)top * 0x10001u;
        const uint32_t spare = (uint32_t)(SS_WINDOW + lane) * 0x10001u;
        for_units([&](int, const uint32_t(&d)[U][4]) {
          const Unpack un;
#pragma unroll
          for (int u = 0; u < U; ++u)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              const uint32_t b = ss_bins(un.keys(d[u][q]), top2, spare);
              atomicAdd(&bins[b & 0xffffu], 1u);
              atomicAdd(&bins[b >> 16], 1u);
            }
        });
        __syncthreads();
      }
      // thread t takes the keys top - (per t + i), i < per, in order
      const int per = (width + SS_THREADS - 1) / SS_THREADS;
      const int b0 = min(tid * per, width), b1 = min(b0 + per, width);
      uint32_t n = 0;
      float w = 0.0f;
      for (int b = b0; b < b1; ++b) {
        const uint32_t c = bins[b];
        if (c) {
          n += c;
          w += (float)c * weight(bf16_key_val((uint32_t)(top - b)));
        }
      }
      // inclusive sums over the wave, then over the waves before it
      const uint32_t sn = sr_scan(n);
      const float sw = sr_scan(w);
      if (lane == 63) {
        wave_n[wave] = sn;
        wave_w[wave] = sw;
      }
      __syncthreads();
      uint32_t all_n = seen_n, base_n = 0;
      float all_w = seen_w, base_w = 0.0f;
#pragma unroll
      for (int v = 0; v < SS_WAVES; ++v) {
        if (v == wave) {
          base_n = all_n;
          base_w = all_w;
        }
        all_n += wave_n[v];
        all_w += wave_w[v];
      }
      {
        uint32_t cn = base_n + sn - n;
        float cw = base_w + sw - w;
        const bool end_k = do_k && cn + n >= (uint32_t)k;
        const bool end_p = do_p && base_w + sw >= target_p;
        if (n && (end_k || end_p)) {   // as above
          int reached = -1;
          for (int b = b0; b < b1; ++b) {
            const uint32_t c = bins[b];
            if (!c) continue;
            cn += c;
            cw += (float)c * weight(bf16_key_val((uint32_t)(top - b)));
            reached = top - b;
            if ((do_k && cn >= (uint32_t)k) || (do_p && cw >= target_p)) break;
          }
          atomicMax(&s_tau, reached);
        }
      }
      __syncthreads();
      tau = s_tau;
      if (tau >= 0) {
        if (some) listed = s_list;
        break;
      }
      if (counted) {   // below what was counted: from the top, all logits
        counted = some = false;
        top = max_key;
        width = SS_WINDOW;
        __syncthreads();
        continue;
      }
      // the highest key below the window
      const int lo = top - width + 1;
      int next = -1;
      for (int at = tid * 8; at < V; at += SS_THREADS * 8) {
        uint32_t d[4];
        load_chunk(at, d);
        const Unpack un;
        for (int q = 0; q < 4; ++q) {
          const uint32_t key = un.keys(d[q]);
          const int k0 = (int)un.first(key), k1 = (int)un.second(key);
          if (k0 < lo) next = max(next, k0);
          if (k1 < lo) next = max(next, k1);
        }
      }
      if (next >= 0) atomicMax(&s_top, next);
      __syncthreads();
      top = s_top;
      seen_n = all_n;
      seen_w = all_w;
      if (top < 0) {  // everything is kept (p * Z not reached by rounding)
        tau = 0;
        break;
      }
      __syncthreads();  // s_top and the bins are reset above
    }
  }

  const uint32_t utau = (uint32_t)tau;
  auto kept = [&](uint32_t key) {
    return key >= utau ? weight(bf16_key_val(key)) : 0.0f;
  };
  auto kept_sum = [&](const uint32_t* e) {
    float sum = 0.0f;
    for (int q = 0; q < 4; ++q) sum += kept(e[q] & 0xffffu) + kept(e[q] >> 16);
    return sum;
  };
  // the element of a chunk at which the running sum passes, or the last with
  // mass
  auto element = [&](const uint32_t* e, float run, float target) {
    int chosen = 0;
    for (int h = 0; h < 8; ++h) {
      const float w = kept((h & 1) ? e[h >> 1] >> 16 : e[h >> 1] & 0xffffu);
      run += w;
      if (w > 0.0f) chosen = h;
      if (w > 0.0f && run > target) break;
    }
    return chosen;
  };

  // ---- listed: at most as many kept chunks as threads are put in order ----
  if (listed >= 0) {
    const Unpack un;
    auto keys_of = [&](int e, uint32_t (&l)[4]) {
      const uint4 v = list_k[e];
      l[0] = un.keys(v.x); l[1] = un.keys(v.y);
      l[2] = un.keys(v.z); l[3] = un.keys(v.w);
    };
    // kept_e and kept_w lie where counts were: nobody reads them any more
    __syncthreads();
    for (int e = tid; e < listed; e += SS_THREADS) {
      uint32_t l[4];
      keys_of(e, l);
      if (largest_key(l) >= utau) {
        const int at = atomicAdd(&s_kept, 1);
        if (at < SS_THREADS) {
          kept_at[at] = list_at[e];
          kept_w[at] = kept_sum(l);
          kept_e[at] = e;
        }
      }
    }
    __syncthreads();
    const int n = s_kept;
    auto rank_of = [&](int own) {
      int rank = 0;
      for (int e = 0; e < n; e += 4) {
        const int4 v = *reinterpret_cast<const int4*>(kept_at + e);
        rank += (v.x < own) + (v.y < own) + (v.z < own) + (v.w < own);
      }
      return rank;
    };
    auto draw = [&](int e, float run, float target) {
      uint32_t l[4];
      keys_of(e, l);
      out[seq] = list_at[e] * 8 + element(l, run, target);
    };
    if (n <= 64) {   // one wave
      if (wave == 0) {
        if (lane < n) {
          const int rank = rank_of(kept_at[lane]);
          sorted_w[rank] = kept_w[lane];
          sorted_e[rank] = kept_e[lane];
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
        __builtin_amdgcn_wave_barrier();
        const float w = lane < n ? sorted_w[lane] : 0.0f;
        const float own = sr_scan(w);
        const float total =
            __builtin_bit_cast(float, __builtin_amdgcn_readlane(
                                          __builtin_bit_cast(int, own), 63));
        if (total > 0.0f) {
          const float target = u01 * total;
          const uint64_t past = __ballot(w > 0.0f && own > target);
          const uint64_t any = __ballot(w > 0.0f);
          const int l = past ? __builtin_ctzll(past) : 63 - __builtin_clzll(any);
          if (lane == l)
            draw(sorted_e[lane], own - w, past ? target : INFINITY);
        } else if (lane == 0) {
          s_last = 1;   // nothing to draw from
        }
      }
      __syncthreads();
      if (s_last == 1) first_max();
      return;
    }
    if (n <= SS_THREADS) {
      if (tid < n) {
        const int rank = rank_of(kept_at[tid]);
        sorted_w[rank] = kept_w[tid];
        sorted_e[rank] = kept_e[tid];
      }
      __syncthreads();
      const float w = tid < n ? sorted_w[tid] : 0.0f;
      const float own = sr_scan(w);
      if (lane == 63) wave_w[wave] = own;
      __syncthreads();
      float before = 0.0f, total = 0.0f;
#pragma unroll
      for (int v = 0; v < SS_WAVES; ++v) {
        if (v == wave) before = total;
        total += wave_w[v];
      }
      if (total > 0.0f) {
        const float target = u01 * total;
        if (w > 0.0f) {
          if (before + own > target) atomicMin(&s_cell, tid);
          atomicMax(&s_last, tid);
        }
        __syncthreads();
        const bool passed = s_cell != INT_MAX;
        if (tid == (passed ? s_cell : s_last))
          draw(sorted_e[tid], before + own - w, passed ? target : INFINITY);
      } else {   // as below
        first_max();
      }
      return;
    }
  }

  // ---- kept mass of every unit, in index order ----
  if (do_list || bad) {
    for_units([&](int unit, const uint32_t(&d)[U][4]) {
      const Unpack un;
      float sum = 0.0f;
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const uint32_t key = un.keys(d[u][q]);
          const float w0 = weight(un.lo(d[u][q])), w1 = weight(un.hi(d[u][q]));
          sum += (un.first(key) >= utau ? w0 : 0.0f) +
                 (un.second(key) >= utau ? w1 : 0.0f);
        }
      sum = sr_sum(sum);
      if (lane == 0) {
        cells[unit] = sum;
        cell_c[unit] = 0.0f;
      }
    });
    __syncthreads();
  }
  // every wave: the first unit whose running sum passes u * total
  constexpr int PER = SS_UNITS / 64;
  float mass[PER], own = 0.0f;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int c = lane * PER + i;
    mass[i] = do_list || bad ? (c < units ? cells[c] : 0.0f) : cell(c);
    own += mass[i];
  }
  float run = sr_scan(own);
  const float total = __shfl(run, 63, 64);
  const float target = u01 * total;
  run -= own;
  int at = -1;         // first that passes the target
  int last = -1;       // last with any mass
  float base = 0.0f;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int c = lane * PER + i;
    const float w = mass[i];
    if (w > 0.0f) last = c;
    if (at < 0 && w > 0.0f && run + w > target) {
      at = c;
      base = run;
    }
    run += w;
  }
  const uint64_t found = __ballot(at >= 0), some = __ballot(last >= 0);
  float rest = INFINITY;   // mass into the unit; infinite: its last element
  int pick = -1;
  if (!(total > 0.0f)) {
    // nothing that could be drawn from: the largest logit
  } else if (found) {
    const int l = __builtin_ctzll(found);
    pick = __shfl(at, l, 64);
    rest = target - __shfl(base, l, 64);
  } else if (some) {
    pick = __shfl(last, 63 - __builtin_clzll(some), 64);
  }
  if (pick < 0) {
    // A kept logit that is not a number, or an infinite one, leaves no mass
    // to draw from: the largest logit, the first one where none is above
    // minus infinity.
    first_max();
    return;
  }
  if (wave != 0) return;
  uint32_t d[U][4];
  load(pick, d);
  float before = 0.0f, at_run = 0.0f;
  int chunk = -1, at_lane = 0;
  bool passed = false;
#pragma unroll
  for (int u = 0; u < U; ++u) {
#pragma unroll
    for (int q = 0; q < 4; ++q) d[u][q] = Unpack().keys(d[u][q]);
    const float sum = kept_sum(d[u]);
    const float to = before + sr_scan(sum);
    const uint64_t past = __ballot(sum > 0.0f && to > rest);
    const uint64_t any = __ballot(sum > 0.0f);
    if (!passed && any) {
      passed = past != 0;
      chunk = u;
      at_lane = past ? __builtin_ctzll(past) : 63 - __builtin_clzll(any);
      at_run = to - sum;
    }
    before = __shfl(to, 63, 64);
  }
  if (lane == at_lane) {
    uint32_t e[4] = {0, 0, 0, 0};
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (u == chunk) {
#pragma unroll
        for (int q = 0; q < 4; ++q) e[q] = d[u][q];
      }
    out[seq] = pick * UNIT + chunk * 512 + lane * 8 +
               element(e, at_run, passed ? rest : INFINITY);
  }
}

void sample(torch::Tensor out, torch::Tensor logits, torch::Tensor temperature,
            torch::Tensor top_k, torch::Tensor top_p, torch::Tensor uniforms) {
  TORCH_CHECK(logits.is_cuda());
  TORCH_CHECK(logits.is_contiguous());
  TORCH_CHECK(out.dtype() == torch::kInt32);
  const int B = logits.size(0);
  const int V = logits.size(1);
  constexpr int BLOCK = 256;
  hipStream_t stream = at::cuda::getCurrentCUDAStream();
  if (logits.dtype() == torch::kBFloat16) {
    if (B == 0) return;
#define LAUNCH_RESIDENT(NCH)                                                  \
  hipLaunchKernelGGL((sample_bf16_resident_kernel<NCH>), dim3(B),             \
                     dim3(SR_THREADS), 0, stream, (int32_t*)out.data_ptr(),   \
                     (const uint16_t*)logits.data_ptr(),                      \
                     (const float*)temperature.data_ptr(),                    \
                     (const int32_t*)top_k.data_ptr(),                        \
                     (const float*)top_p.data_ptr(),                          \
                     (const float*)uniforms.data_ptr(), V)
    // Longer rows than the resident kernel is ahead for (its line: see there), up
    // to what `cells` holds.  Up to a row per compute unit, 1024 threads a row: 64
    // and 400 rows of 128256, mixed requests, 39.9 and 61.8 us, with 512 threads
    // and two rows on a unit 42.3 and 57.8.
    if (V > 16 * 8 * SR_THREADS && V <= SS_UNITS * SS_UNIT) {
#define LAUNCH_STREAM(T)                                                      \
  hipLaunchKernelGGL((sample_bf16_stream_kernel<T>), dim3(B), dim3(T), 0,     \
                     stream, (int32_t*)out.data_ptr(),                        \
                     (const uint16_t*)logits.data_ptr(),                      \
                     (const float*)temperature.data_ptr(),                    \
                     (const int32_t*)top_k.data_ptr(),                        \
                     (const float*)top_p.data_ptr(),                          \
                     (const float*)uniforms.data_ptr(), V,                    \
                     B > 512 && B <= SS_ORDERED)
      if (B <= 256) LAUNCH_STREAM(1024);
      else LAUNCH_STREAM(512);
#undef LAUNCH_STREAM
      HIP_CHECK_KERNEL();
      return;
    }
    const int chunks = (V + 8 * SR_THREADS - 1) / (8 * SR_THREADS);
    if (V > 8 * SR_THREADS && chunks <= 16) {
      if (chunks <= 2) LAUNCH_RESIDENT(2);
      else if (chunks <= 4) LAUNCH_RESIDENT(4);
      else if (chunks <= 6) LAUNCH_RESIDENT(6);
      else if (chunks <= 8) LAUNCH_RESIDENT(8);
      else if (chunks <= 12) LAUNCH_RESIDENT(12);
      else LAUNCH_RESIDENT(16);
      HIP_CHECK_KERNEL();
      return;
    }
#undef LAUNCH_RESIDENT
    // 8 waves per row: the radix walk is latency-bound at 4 waves
    // (PMC: 50% parked / 32% issue-stalled at BLOCK=256)
    constexpr int BLOCK_BF16 = 512;
    hipLaunchKernelGGL((sample_bf16_kernel<BLOCK_BF16>), dim3(B),
                       dim3(BLOCK_BF16), 0,
                       stream, (int32_t*)out.data_ptr(),
                       (const uint16_t*)logits.data_ptr(),
                       (const float*)temperature.data_ptr(),
                       (const int32_t*)top_k.data_ptr(),
                       (const float*)top_p.data_ptr(),
                       (const float*)uniforms.data_ptr(), V);
    HIP_CHECK_KERNEL();
    return;
  }
  TORCH_CHECK(logits.dtype() == torch::kFloat32);
  hipLaunchKernelGGL((sample_kernel<BLOCK>), dim3(B), dim3(BLOCK), 0, stream,
                     (int32_t*)out.data_ptr(), (const float*)logits.data_ptr(),
                     (const float*)temperature.data_ptr(),
                     (const int32_t*)top_k.data_ptr(),
                     (const float*)top_p.data_ptr(),
                     (const float*)uniforms.data_ptr(), V);
  HIP_CHECK_KERNEL();
}

}  // namespace igw
