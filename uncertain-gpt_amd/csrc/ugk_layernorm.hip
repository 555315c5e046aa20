// ugk_layernorm.hip - LayerNorm forward and backward (train_bnn.c:81-115,
// :439-477), and the residual -> LayerNorm / LayerNorm -> residual pairs of
// the reference launch sequence fused into one pass each.
//
// Layout: rows of C fp32 values, row-major; mean/rstd one float per row;
// weight/bias/dweight/dbias C floats.
//
// Forward: one wavefront per row. Each lane holds V float4 of the row in
// registers (V = ceil(C/256); C = 768 -> 3), so the row is read from HBM once
// and written once (8 bytes per element). Mean and variance are two-pass over
// the registers with wavefront sums (DPP within rows of 16 lanes, the four
// row sums added in scalar registers), rstd = 1/sqrtf(var/C + 1e-5) with IEEE
// division and square root, exactly the CPU formula.
//
// Backward: one wavefront per row for dinp (two wavefront sums). Each
// wavefront adds the dweight/dbias terms of its rows, in row order, in
// registers; after one barrier the workgroup's W per-wavefront sums are added
// column by column in wavefront order into one partial row per workgroup, and
// a second, small kernel adds the partial rows in a fixed order into
// dweight/dbias. No atomics, so the result is identical run to run.
//
// The float4 paths take rows at any alignment (gfx950 accepts a 16-byte access
// at a 4-byte address) and widths that are no multiple of 4, whose last slot
// overlaps the one before it (Cols). Every load of theirs is unconditional: a
// lane's columns past the row are clamped onto the row's last four floats, and
// rows past a wavefront's range repeat its last row; the values so loaded are masked out of the sums
// (added as -0.0f, the identity of IEEE addition) or skipped by a branch that
// is uniform across the wavefront, and never stored. Per-lane
// conditions around loads made the compiler wait for one row's loads before
// it issued the next row's.
// Streamed rows (x, dout, dinp, out) use non-temporal loads and stores.
#include <algorithm>
#include <atomic>
#include <mutex>

#include "ugk_internal.h"

namespace ugk {
namespace {

constexpr int kWavesPerBlock = kBlock / kWave;
constexpr int kMaxV = 8;  // float4 per lane held in registers: C <= 2048
constexpr int kMaxWide = 8192;  // channels of the workgroup-per-row kernels

__device__ __forceinline__ float4 add4(float4 a, float4 b) {
  return make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w);
}

// A lane's V slots of four columns in a row: the slot's first float and the
// components that are the slot's own, [lo, 4). Slots past the row repeat its
// last four floats (lo = 4). With C no multiple of 4 (kRag) the last slot
// does so too, for the components that the slot before it does not hold; they
// are loaded twice and summed and stored once. C >= 4.
template <int V, bool kRag>
struct Cols {
  int at[V], lo[V];
  // slot v of the lane is slot first + v * step of the row
  __device__ __forceinline__ Cols(int first, int step, int C) {
#pragma unroll
    for (int v = 0; v < V; v++) {
      const int c = 4 * (first + v * step);
      at[v] = min(c, C - 4);
      lo[v] = kRag ? min(c - at[v], 4) : c < C ? 0 : 4;
    }
  }
  // component j of slot v is the slot's own
  __device__ __forceinline__ bool own(int v, int j) const { return kRag ? j >= lo[v] : lo[v] == 0; }
  __device__ __forceinline__ bool any(int v) const { return lo[v] < 4; }
  // x where own, else the identity of IEEE addition
  __device__ __forceinline__ float sel(int v, int j, float x) const { return own(v, j) ? x : -0.0f; }
  // non-temporal store of the slot's own components to row + at[v]
  __device__ __forceinline__ void put(float *row, int v, float4 x) const {
    float *p = row + at[v];
    if (lo[v] == 0) {
      st_nt4(p, x);
    } else if (kRag) {
      if (lo[v] <= 1) st_nt(p + 1, x.y);
      if (lo[v] <= 2) st_nt(p + 2, x.z);
      if (lo[v] <= 3) st_nt(p + 3, x.w);
    }
  }
};

// Row statistics to outputs: v = (x - m) r w + b.
__device__ __forceinline__ float4 ln_norm4(float4 x, float m, float r, float4 w, float4 b) {
  return make_float4((x.x - m) * r * w.x + b.x, (x.y - m) * r * w.y + b.y, (x.z - m) * r * w.z + b.z,
                     (x.w - m) * r * w.w + b.w);
}

// A lane's share of a row's sum, and of the sum of its squared distances from m.
template <int V, bool kRag>
__device__ __forceinline__ float ln_lane_sum(const float4 (&xv)[V], const Cols<V, kRag> &cl) {
  float s = 0.0f;
#pragma unroll
  for (int v = 0; v < V; v++) {
    s += cl.sel(v, 0, xv[v].x); s += cl.sel(v, 1, xv[v].y); s += cl.sel(v, 2, xv[v].z); s += cl.sel(v, 3, xv[v].w);
  }
  return s;
}
template <int V, bool kRag>
__device__ __forceinline__ float ln_lane_sq(const float4 (&xv)[V], const Cols<V, kRag> &cl, float m) {
  float vs = 0.0f;
#pragma unroll
  for (int v = 0; v < V; v++) {
    float d;
    d = xv[v].x - m; vs += cl.sel(v, 0, d * d);
    d = xv[v].y - m; vs += cl.sel(v, 1, d * d);
    d = xv[v].z - m; vs += cl.sel(v, 2, d * d);
    d = xv[v].w - m; vs += cl.sel(v, 3, d * d);
  }
  return vs;
}

// Normalise one row held in registers (V float4 per lane) and store out, mean
// and rstd: two-pass mean and variance with wavefront sums, IEEE 1/sqrtf.
// Shared by every one-wavefront forward kernel, so that they give the same bits.
// kEarly: weight and bias are loaded before the sums rather than where they are
// used, one round trip to the cache off the row's chain. It pays while the
// rows leave the SIMDs idle for that long (residual and forward at 1,024 x 768
// 4.3 against 4.6 us, 512 x 1,600 5.1 against 5.8), not for its registers beyond
// (8,192 x 768 18.6 against 18.2).
template <int V, bool kRag, bool kEarly>
__device__ __forceinline__ void ln_row_out(const float4 (&xv)[V], const Cols<V, kRag> &cl, int C, int row, int lane,
                                           const float *__restrict__ weight, const float *__restrict__ bias,
                                           float *__restrict__ out, float *__restrict__ mean,
                                           float *__restrict__ rstd) {
  float4 w[kEarly ? V : 1], b[kEarly ? V : 1];
  if constexpr (kEarly) {
#pragma unroll
    for (int v = 0; v < V; v++) {
      w[v] = ld4(weight + cl.at[v]);
      b[v] = ld4(bias + cl.at[v]);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  const float m = wave_sum(ln_lane_sum(xv, cl)) / (float)C;
  const float r = 1.0f / sqrtf(wave_sum(ln_lane_sq(xv, cl, m)) / (float)C + 1e-5f);
  float *o = out + (size_t)row * C;
#pragma unroll
  for (int v = 0; v < V; v++)
    if (cl.any(v)) {
      if constexpr (kEarly)
        cl.put(o, v, ln_norm4(xv[v], m, r, w[v], b[v]));
      else
        cl.put(o, v, ln_norm4(xv[v], m, r, ld4(weight + cl.at[v]), ld4(bias + cl.at[v])));
    }
  if (lane == 0) {
    mean[row] = m;
    rstd[row] = r;
  }
}

// Forward, RPW rows per wavefront (consecutive). The loads of row k+1 are
// issued before row k is normalised and stored, so a wavefront has a row in
// flight while it writes one.
// kRes: the row is first formed as res = inp + inp2 (residual_forward,
// train_bnn.c:182-186), stored to res, and normalised from the registers, the
// pair gpt2_kernels.cuh:793-797 launches back to back.
template <int V, bool kRes, int RPW, bool kRag, bool kEarly>
__global__ __launch_bounds__(kBlock) void k_ln_fwd_vec(float *__restrict__ out, float *__restrict__ mean,
                                                       float *__restrict__ rstd, const float *__restrict__ inp,
                                                       const float *__restrict__ weight,
                                                       const float *__restrict__ bias, int rows, int C,
                                                       float *__restrict__ res, const float *__restrict__ inp2) {
  const int lane = threadIdx.x & (kWave - 1);
  const int row0 = (blockIdx.x * kWavesPerBlock + (threadIdx.x >> 6)) * RPW;
  if (row0 >= rows) return;
  const Cols<V, kRag> cl(lane, kWave, C);
  float4 xa[V], ya[kRes ? V : 1];
  {
    const size_t off = (size_t)row0 * C;
#pragma unroll
    for (int v = 0; v < V; v++) {
      xa[v] = ld_nt4(inp + off + cl.at[v]);
      if (kRes) ya[kRes ? v : 0] = ld_nt4(inp2 + off + cl.at[v]);
    }
  }
#pragma unroll
  for (int k = 0; k < RPW; k++) {
    const int row = row0 + k;
    if (row >= rows) break;
    float4 xb[V], yb[kRes ? V : 1];
    if (k + 1 < RPW) {
      const size_t off = (size_t)min(row + 1, rows - 1) * C;
#pragma unroll
      for (int v = 0; v < V; v++) {
        xb[v] = ld_nt4(inp + off + cl.at[v]);
        if (kRes) yb[kRes ? v : 0] = ld_nt4(inp2 + off + cl.at[v]);
      }
    }
    float4 xv[V];
#pragma unroll
    for (int v = 0; v < V; v++) {
      xv[v] = xa[v];
      if (kRes) {
        xv[v] = add4(xv[v], ya[kRes ? v : 0]);
        cl.put(res + (size_t)row * C, v, xv[v]);
      }
    }
    ln_row_out<V, kRag, kEarly>(xv, cl, C, row, lane, weight, bias, out, mean, rstd);
    if (k + 1 < RPW) {
#pragma unroll
      for (int v = 0; v < V; v++) {
        xa[v] = xb[v];
        if (kRes) ya[kRes ? v : 0] = yb[kRes ? v : 0];
      }
    }
  }
}

// Encoder forward then LayerNorm forward of its output, RPW rows per
// wavefront: row (b, t) is formed as wte[inp[b,t]] + wpe[t] in registers (the
// single add of train_bnn.c:41-65, the encoder's own order), stored to enc,
// and normalised from the registers as k_ln_fwd_vec does: the pair
// gpt2_kernels.cuh:775 -> :784 (or :813 when L = 0) launches back to back.
// The rows of wte and wpe are read through the cache: tokens repeat, and the
// B rows of a position share its wpe row.
template <int V, int RPW, bool kEarly>
__global__ __launch_bounds__(kBlock) void k_enc_ln_fwd_vec(float *__restrict__ enc, float *__restrict__ out,
                                                           float *__restrict__ mean, float *__restrict__ rstd,
                                                           int *inp, IdCheck ids,
                                                           const float *__restrict__ wte,
                                                           const float *__restrict__ wpe,
                                                           const float *__restrict__ weight,
                                                           const float *__restrict__ bias, int rows, int T, int C) {
  const int lane = threadIdx.x & (kWave - 1);
  const int row0 = (blockIdx.x * kWavesPerBlock + (threadIdx.x >> 6)) * RPW;
  if (row0 >= rows) return;
  const Cols<V, false> cl(lane, kWave, C);
  float4 xa[V], ya[V];
  // every id of the wavefront, and the first row of wpe, on their way before the
  // first check: its branch, and the store in it, would hold back what comes after
  int id[RPW];
#pragma unroll
  for (int k = 0; k < RPW; k++) id[k] = inp[min(row0 + k, rows - 1)];
  {
    const float *pe = wpe + (size_t)(row0 % T) * C;
#pragma unroll
    for (int v = 0; v < V; v++) ya[v] = ld4(pe + cl.at[v]);
    const int ix = check_id(__builtin_amdgcn_readfirstlane(id[0]), inp, row0, ids);
    const float *te = wte + (size_t)ix * C;
#pragma unroll
    for (int v = 0; v < V; v++) xa[v] = ld4(te + cl.at[v]);
  }
#pragma unroll
  for (int k = 0; k < RPW; k++) {
    const int row = row0 + k;
    if (row >= rows) break;
    float4 xb[V], yb[V];
    if (k + 1 < RPW) {
      const int nx = min(row + 1, rows - 1);
      const int ix = check_id(__builtin_amdgcn_readfirstlane(id[k + 1 < RPW ? k + 1 : k]), inp, nx, ids);
      const float *te = wte + (size_t)ix * C, *pe = wpe + (size_t)(nx % T) * C;
#pragma unroll
      for (int v = 0; v < V; v++) {
        xb[v] = ld4(te + cl.at[v]);
        yb[v] = ld4(pe + cl.at[v]);
      }
    }
    float4 xv[V];
#pragma unroll
    for (int v = 0; v < V; v++) {
      xv[v] = add4(xa[v], ya[v]);
      cl.put(enc + (size_t)row * C, v, xv[v]);
    }
    ln_row_out<V, false, kEarly>(xv, cl, C, row, lane, weight, bias, out, mean, rstd);
    if (k + 1 < RPW) {
#pragma unroll
      for (int v = 0; v < V; v++) {
        xa[v] = xb[v];
        ya[v] = yb[v];
      }
    }
  }
}

// Forward for rows of more than 2,048 channels: a workgroup of W wavefronts
// per row, V float4 per lane in registers, so the row is still read once
// (the one-wavefront kernel would need more than 32 registers for it, and the
// lane loop below reads it three times). Each of the row's two sums is a lane
// sum, a wavefront sum and the W wavefronts' sums added in order by every
// thread, one barrier each. Memory-bound: 4,092 x 4,096 in 26.4 us (5.1 TB/s),
// 83 us in the lane loop.
template <int V, int W, bool kRes>
__global__ __launch_bounds__(W * kWave) void k_ln_fwd_wide(float *__restrict__ out, float *__restrict__ mean,
                                                           float *__restrict__ rstd, const float *__restrict__ inp,
                                                           const float *__restrict__ weight,
                                                           const float *__restrict__ bias, int C,
                                                           float *__restrict__ res, const float *__restrict__ inp2) {
  __shared__ float part[2][W];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & (kWave - 1);
  const int row = blockIdx.x;
  const size_t off = (size_t)row * C;
  const Cols<V, true> cl(threadIdx.x, W * kWave, C);
  float4 xv[V], yv[kRes ? V : 1];
#pragma unroll
  for (int v = 0; v < V; v++) {
    xv[v] = ld_nt4(inp + off + cl.at[v]);
    if (kRes) yv[kRes ? v : 0] = ld_nt4(inp2 + off + cl.at[v]);
  }
  if (kRes) {
#pragma unroll
    for (int v = 0; v < V; v++) {
      xv[v] = add4(xv[v], yv[kRes ? v : 0]);
      cl.put(res + off, v, xv[v]);
    }
  }
  const auto row_sum = [&](float mine, float *p) {
    mine = wave_sum(mine);
    if (lane == 0) p[wave] = mine;
    __syncthreads();
    float t = p[0];
#pragma unroll
    for (int k = 1; k < W; k++) t += p[k];
    return t;
  };
  const float m = row_sum(ln_lane_sum(xv, cl), part[0]) / (float)C;
  const float r = 1.0f / sqrtf(row_sum(ln_lane_sq(xv, cl, m), part[1]) / (float)C + 1e-5f);
#pragma unroll
  for (int v = 0; v < V; v++)
    if (cl.any(v)) cl.put(out + off, v, ln_norm4(xv[v], m, r, ld4(weight + cl.at[v]), ld4(bias + cl.at[v])));
  if (threadIdx.x == 0) {
    mean[row] = m;
    rstd[row] = r;
  }
}

// Any C (the rows that no kernel above takes: C < 4 or beyond 8,192): one
// wavefront per row, three passes over the row.
__global__ __launch_bounds__(kBlock) void k_ln_fwd_scalar(float *out, float *mean, float *rstd,
                                                          const float *inp, const float *weight,
                                                          const float *bias, int rows, int C) {
  const int lane = threadIdx.x & (kWave - 1);
  const int row = blockIdx.x * kWavesPerBlock + (threadIdx.x >> 6);
  if (row >= rows) return;
  const float *x = inp + (size_t)row * C;
  float *o = out + (size_t)row * C;
  float s = 0.0f;
  for (int c = lane; c < C; c += kWave) s += x[c];
  s = wave_sum(s);
  const float m = s / (float)C;
  float vs = 0.0f;
  for (int c = lane; c < C; c += kWave) {
    const float d = x[c] - m;
    vs += d * d;
  }
  vs = wave_sum(vs);
  const float r = 1.0f / sqrtf(vs / (float)C + 1e-5f);
  for (int c = lane; c < C; c += kWave) o[c] = (x[c] - m) * r * weight[c] + bias[c];
  if (lane == 0) {
    mean[row] = m;
    rstd[row] = r;
  }
}

__device__ __forceinline__ float4 zero4() { return make_float4(0.0f, 0.0f, 0.0f, 0.0f); }

// ---- column sums in the main launch (the per-op entry points) ----------------
// Instead of a second launch over the partial rows, the workgroups finish the
// column sums themselves, in the order the column-sum kernel uses (so with the
// same bits): the partial rows form kTailGroups groups of J = ceil(nblk / 16)
// consecutive rows; the last workgroup of a group to finish adds the group's
// rows (RowChains) and writes the sum over the group's first row; the last group to finish adds the group sums in group
// order (an empty group adds +0.0f) into dweight/dbias.
//
// Publishing without a cache write-back: the rows and group sums are written
// with device-scope stores (sc1: written through to the point where all of the
// device's L2 caches are coherent) and read with device-scope loads. Each
// thread waits for its own stores to complete (s_waitcnt vmcnt(0)) before the
// workgroup barrier after which one thread increments the group's counter (a
// device-scope atomic), so when a counter shows a workgroup that it is the
// last, every row it is about to read is already at the coherence point. This
// is the release/acquire pair that an agent-scope fence would implement with
// an L2 write-back (buffer_wbl2 sc1) and invalidation on gfx950, confined to
// the bytes that need it; the fence itself, once per workgroup, took the call
// from 23 to 180 us at 8,192 x 768. Without it the call still takes longer
// than with the second launch (32.7 against 23.3 us at 8,192 x 768, 108
// against 38 us at 4,096 x 2,048): the last workgroup's chain of dependent
// device-scope round trips (its stores' completion, the counter, the group's
// rows, the group sum's completion, the counter, the group sums), about
// 0.85 us each, outlasts a launch that needs two. So it is not the default
// (ugk_diag_layernorm_tail selects it).
//
// The counters are per device and zero when the code object is loaded; the
// last arriver of each level resets its counter, so every call finds them at
// zero. Calls that overlap on one device (other streams) would share them,
// as they would share the workspace.
constexpr int kTailGroups = 16;
}  // namespace
}  // namespace ugk

static __device__ int ln_tail_count[ugk::kTailGroups + 1];

namespace ugk {
namespace {

__device__ __forceinline__ void st_dev(float *p, float v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float ld_dev(float *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ void wait_stores() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// A column's sum over the partial rows of a group: four chains, every fourth
// row to each, in index order, then the chains in pairs. One chain of up to 64
// rows is further from the 64-bit sums the more partial rows a call has:
// dweight of 15,345 x 768 (959 partial rows) was 1.75e-7 off with one chain (in
// the 2-norm, relative) and is 1.33e-7 off with four, at the same time.
struct RowChains {
  float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  // the next rows of the group, `left` of them up to its end
  template <int N>
  __device__ __forceinline__ void add(const float (&v)[N], int left) {
    static_assert(N % 4 == 0, "a batch starts on the first chain");
#pragma unroll
    for (int q = 0; q < N; q++) s[q & 3] += q < left ? v[q] : -0.0f;
  }
  __device__ __forceinline__ float sum() const { return (s[0] + s[1]) + (s[2] + s[3]); }
};

// Called by every thread of a workgroup (NT threads) after it has written its
// partial row with st_dev.
template <int NT>
__device__ __forceinline__ void ln_bwd_tail(float *partial, int nblk, int C, float *dweight, float *dbias) {
  __shared__ int last;
  constexpr int kBatch = 16;
  const int C2 = 2 * C;
  const int J = (nblk + kTailGroups - 1) / kTailGroups;
  const int g = blockIdx.x / J;
  const int j0 = g * J, j1 = min(j0 + J, nblk);
  wait_stores();
  __syncthreads();
  if (threadIdx.x == 0) {
    const int old = __hip_atomic_fetch_add(&ln_tail_count[g], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    last = old == j1 - j0 - 1;
    if (last) __hip_atomic_store(&ln_tail_count[g], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  if (!last) return;
  for (int c = threadIdx.x; c < C2; c += NT) {
    RowChains acc;
    for (int b = j0; b < j1; b += kBatch) {
      float v[kBatch];
#pragma unroll
      for (int q = 0; q < kBatch; q++) v[q] = ld_dev(partial + (size_t)min(b + q, j1 - 1) * C2 + c);
      acc.add(v, j1 - b);
    }
    st_dev(partial + (size_t)j0 * C2 + c, acc.sum());
  }
  wait_stores();
  __syncthreads();
  const int G = (nblk + J - 1) / J;  // groups with rows
  if (threadIdx.x == 0) {
    const int old = __hip_atomic_fetch_add(&ln_tail_count[kTailGroups], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    last = old == G - 1;
    if (last) __hip_atomic_store(&ln_tail_count[kTailGroups], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  if (!last) return;
  for (int c = threadIdx.x; c < C2; c += NT) {
    float v[kTailGroups];
#pragma unroll
    for (int k = 0; k < kTailGroups; k++) v[k] = ld_dev(partial + (size_t)min(k, G - 1) * J * C2 + c);
    float t = v[0];
#pragma unroll
    for (int k = 1; k < kTailGroups; k++) t += k < G ? v[k] : 0.0f;
    if (c < C)
      dweight[c] += t;
    else
      dbias[c - C] += t;
  }
}

// Backward, register-resident rows. A workgroup is W wavefronts; wavefront w
// of workgroup g takes the rpw consecutive rows starting at (W g + w) * rpw,
// R at a time: the loads of R rows (x and dout first, which the row sums
// need, then dinp and the residual rows) are all issued before the first
// arithmetic instruction. It writes dinp and adds its rows' dweight/dbias
// terms, in row order, into its registers. After one barrier, thread t of the
// workgroup adds float4 column t of the W wavefronts' sums in wavefront order
// and writes the workgroup's partial row:
// partial[g] = [dweight part (C floats) | dbias part (C floats)].
// The weight row is read from global memory (it stays in L2), so the first
// rows' loads go out without waiting for anything.
//
// kRes: the new dinp row is also added to rdx and rdy (residual_backward with
// dout = dinp, train_bnn.c:491-496; twice into rdx when same), the pair
// gpt2_kernels.cuh:870-876 launches back to back.
// kDinp: kDinpRw reads and writes dinp. kDinpRead (kRes only) reads it but
// does not write it back: the step driver's pairs, whose dinp nothing reads
// after the residual split. kDinpNone (kRes only) neither reads nor writes
// it, taking it as +0.0: the first pair of the zeroed-gradient driver.
// kAssign (kRes only): rdx and rdy are not read but taken as +0.0 (the
// zeroed-gradient driver, whose residual targets are first written there).
// +0.0 + x is x with -0.0 turned to +0.0, so both give the bits the reads
// would give on a zero buffer.
// MINW: wavefronts per SIMD the register allocation must allow.
// kNt: dinp is written with non-temporal stores (always with kRes). Without
// kRes, large calls write it with ordinary stores, which measured faster
// (8,192 x 768: 17.5 against 19.0 us in the step, 22.7 against 23.9 us with
// the column sums); below 2^21 elements, where the written rows fit the
// caches and are written back at the end of the launch, non-temporal stores
// are kept. The fused pair keeps non-temporal stores for all three rows:
// an ordinary dinp store made it faster alone (35.7 against 37.2 us cold at
// 8,192 x 768) but the step slower (3.02 against 2.93 ms), the dirty lines
// of its 24 launches being written back during the kernels that follow.
template <int V, int W, int R, bool kRes, int MINW, bool kNt, int kDinp, bool kAssign, bool kTail, bool kRag>
__global__ __launch_bounds__(W * kWave, MINW) void k_ln_bwd_vec(
    float *__restrict__ dinp, float *__restrict__ partial, const float *__restrict__ dout,
    const float *__restrict__ inp, const float *__restrict__ weight, const float *__restrict__ mean,
    const float *__restrict__ rstd, int rows, int C, int rpw, float *__restrict__ rdx,
    float *__restrict__ rdy, int same, float *dweight, float *dbias) {
  static_assert(!kRag || (kNt && !kTail), "ragged rows take the non-temporal stores and the second launch");
  __shared__ float4 red[W][2][V * kWave];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x >> 6;
  const float Cf = (float)C;
  const Cols<V, kRag> cl(lane, kWave, C);
  float4 ag[V], ab[V];
#pragma unroll
  for (int v = 0; v < V; v++) ag[v] = ab[v] = make_float4(0.f, 0.f, 0.f, 0.f);
  const int row0 = (blockIdx.x * W + wave) * rpw;
  const int row1 = min(row0 + rpw, rows);
  for (int row = row0; row < row1; row += R) {
    const int nr = min(R, row1 - row);
    int rq[R];
    size_t off[R];
#pragma unroll
    for (int q = 0; q < R; q++) {
      rq[q] = row + min(q, nr - 1);
      off[q] = (size_t)rq[q] * C;
    }
    float4 x[R][V], dy[R][V], dx[R][V], wv[V];
    float4 ra[kRes ? R : 1][kRes ? V : 1], rb[kRes ? R : 1][kRes ? V : 1];
    float m[R], r[R];
#pragma unroll
    for (int q = 0; q < R; q++)
#pragma unroll
      for (int v = 0; v < V; v++) x[q][v] = ld_nt4(inp + off[q] + cl.at[v]);
#pragma unroll
    for (int q = 0; q < R; q++)
#pragma unroll
      for (int v = 0; v < V; v++) dy[q][v] = ld_nt4(dout + off[q] + cl.at[v]);
#pragma unroll
    for (int v = 0; v < V; v++) wv[v] = ld4(weight + cl.at[v]);
#pragma unroll
    for (int q = 0; q < R; q++) {
      m[q] = mean[rq[q]];
      r[q] = rstd[rq[q]];
    }
#pragma unroll
    for (int q = 0; q < R; q++)
#pragma unroll
      for (int v = 0; v < V; v++) dx[q][v] = kDinp == kDinpNone ? zero4() : ld_nt4(dinp + off[q] + cl.at[v]);
    if (kRes) {
      // rdy is loaded even when it is rdx (same): a valid address, never used
#pragma unroll
      for (int q = 0; q < R; q++)
#pragma unroll
        for (int v = 0; v < V; v++) {
          ra[kRes ? q : 0][kRes ? v : 0] = kAssign ? zero4() : ld_nt4(rdx + off[q] + cl.at[v]);
          rb[kRes ? q : 0][kRes ? v : 0] = kAssign ? zero4() : ld_nt4(rdy + off[q] + cl.at[v]);
        }
    }
    // keep every load above the arithmetic (the scheduler would otherwise
    // sink the dinp and residual loads past the row sums)
    __builtin_amdgcn_sched_barrier(0);
    float s1[R], s2[R];
#pragma unroll
    for (int q = 0; q < R; q++) {
      s1[q] = 0.0f;
      s2[q] = 0.0f;
#pragma unroll
      for (int v = 0; v < V; v++) {
        const float4 w = wv[v];
        float4 xh, dn;
        xh.x = (x[q][v].x - m[q]) * r[q]; dn.x = dy[q][v].x * w.x;
        xh.y = (x[q][v].y - m[q]) * r[q]; dn.y = dy[q][v].y * w.y;
        xh.z = (x[q][v].z - m[q]) * r[q]; dn.z = dy[q][v].z * w.z;
        xh.w = (x[q][v].w - m[q]) * r[q]; dn.w = dy[q][v].w * w.w;
        s1[q] += cl.sel(v, 0, dn.x); s2[q] += cl.sel(v, 0, dn.x * xh.x);
        s1[q] += cl.sel(v, 1, dn.y); s2[q] += cl.sel(v, 1, dn.y * xh.y);
        s1[q] += cl.sel(v, 2, dn.z); s2[q] += cl.sel(v, 2, dn.z * xh.z);
        s1[q] += cl.sel(v, 3, dn.w); s2[q] += cl.sel(v, 3, dn.w * xh.w);
      }
    }
#pragma unroll
    for (int q = 0; q < R; q++) {
      s1[q] = wave_sum(s1[q]);
      s2[q] = wave_sum(s2[q]);
    }
#pragma unroll
    for (int q = 0; q < R; q++) {
      // The plain backward waits for dinp's loads here, once. Left to itself the
      // compiler waits before each slot's store, counting the stores before it as
      // if they were loads (8,192 x 2,048 59.1 against 57.7 us, 16,384 x 384 23.6
      // against 22.9, 1,100 x 257 8.7 against 8.0; the pair, with more to wait
      // for, is the slower for it at 8,192 x 2,048: 111 against 108).
      if (q == 0 && !kRes) __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
      const bool live = q < nr;  // rows past nr repeat row nr-1: computed, neither stored nor summed
      const float dnm = s1[q] / Cf, dnxm = s2[q] / Cf;
#pragma unroll
      for (int v = 0; v < V; v++) {
        const float4 w = wv[v];
        float4 xh, dn;
        xh.x = (x[q][v].x - m[q]) * r[q]; dn.x = dy[q][v].x * w.x;
        xh.y = (x[q][v].y - m[q]) * r[q]; dn.y = dy[q][v].y * w.y;
        xh.z = (x[q][v].z - m[q]) * r[q]; dn.z = dy[q][v].z * w.z;
        xh.w = (x[q][v].w - m[q]) * r[q]; dn.w = dy[q][v].w * w.w;
        float4 o;
        o.x = dx[q][v].x + r[q] * (dn.x - dnm - xh.x * dnxm);
        o.y = dx[q][v].y + r[q] * (dn.y - dnm - xh.y * dnxm);
        o.z = dx[q][v].z + r[q] * (dn.z - dnm - xh.z * dnxm);
        o.w = dx[q][v].w + r[q] * (dn.w - dnm - xh.w * dnxm);
        if (cl.any(v) && live) {
          if (kDinp == kDinpRw) {
            if (kNt)
              cl.put(dinp + off[q], v, o);
            else
              st4(dinp + off[q] + cl.at[v], o);
          }
          if (kRes) {
            float4 a = add4(ra[kRes ? q : 0][kRes ? v : 0], o);
            if (same) {
              a = add4(a, o);
            } else {
              cl.put(rdy + off[q], v, add4(rb[kRes ? q : 0][kRes ? v : 0], o));
            }
            cl.put(rdx + off[q], v, a);
          }
        }
        if (q > 0 && !live) continue;  // uniform across the wavefront: a branch, not a mask per lane
        ab[v].x += cl.sel(v, 0, dy[q][v].x); ag[v].x += cl.sel(v, 0, dy[q][v].x * xh.x);
        ab[v].y += cl.sel(v, 1, dy[q][v].y); ag[v].y += cl.sel(v, 1, dy[q][v].y * xh.y);
        ab[v].z += cl.sel(v, 2, dy[q][v].z); ag[v].z += cl.sel(v, 2, dy[q][v].z * xh.z);
        ab[v].w += cl.sel(v, 3, dy[q][v].w); ag[v].w += cl.sel(v, 3, dy[q][v].w * xh.w);
      }
    }
  }
#pragma unroll
  for (int v = 0; v < V; v++) {
    red[wave][0][v * kWave + lane] = ag[v];
    red[wave][1][v * kWave + lane] = ab[v];
  }
  __syncthreads();
  float *prow = partial + (size_t)blockIdx.x * 2 * C;
  for (int e = threadIdx.x; e < 2 * V * kWave; e += W * kWave) {
    const int which = e >= V * kWave ? 1 : 0;
    const int c4 = e - which * V * kWave;
    const Cols<1, kRag> cs(c4, 0, C);
    if (cs.any(0)) {
      float4 t = red[0][which][c4];
#pragma unroll
      for (int k = 1; k < W; k++) t = add4(t, red[k][which][c4]);
      float *q = prow + which * C + cs.at[0];
      if (kTail) {
        st_dev(q, t.x); st_dev(q + 1, t.y); st_dev(q + 2, t.z); st_dev(q + 3, t.w);
      } else if (!kRag || cs.lo[0] == 0) {
        st4(q, t);
      } else {
        if (cs.lo[0] <= 1) q[1] = t.y;
        if (cs.lo[0] <= 2) q[2] = t.z;
        if (cs.lo[0] <= 3) q[3] = t.w;
      }
    }
  }
  if (kTail) ln_bwd_tail<W * kWave>(partial, (int)gridDim.x, C, dweight, dbias);
}

// Backward with each row split over a team of P wavefronts, one float4 per
// lane (C/4 <= 64 P). T teams form a workgroup; team t of workgroup g takes the
// rpt consecutive rows starting at (T g + t) * rpt, R at a time, all their
// loads issued before the first arithmetic instruction. Each wavefront adds
// its part of a row's two sums (the four components in order, then a
// wavefront sum) and writes it to LDS; after a barrier every wavefront of the
// team adds the P parts in part order, so all of them hold the same row sums.
// The dweight/dbias terms of a wavefront's columns are added in registers in
// row order; at the end the T teams' sums are added column by column in team
// order into the workgroup's partial row, as in k_ln_bwd_vec. With four rows
// in flight the fused pair needs 155 registers, so a 12-wavefront workgroup
// (P = 3, T = 4) runs alone on a CU: 35.7 against 37.2 us for the
// two-rows-per-wavefront kernel at 8,192 x 768, cold, with the same 512
// partial rows. rpt and T fix the order of every addition; R does not, so the
// plain backward (R = 2) and the fused pair (R = 4) give the same bits.
template <int P, int T, int R, bool kRes, int MINW, bool kNt, int kDinp, bool kAssign, bool kTail>
__global__ __launch_bounds__(P * T * kWave, MINW) void k_ln_bwd_team(
    float *__restrict__ dinp, float *__restrict__ partial, const float *__restrict__ dout,
    const float *__restrict__ inp, const float *__restrict__ weight, const float *__restrict__ mean,
    const float *__restrict__ rstd, int rows, int C, int rpt, float *__restrict__ rdx,
    float *__restrict__ rdy, int same, float *dweight, float *dbias) {
  __shared__ float parts[2][T][R][P][2];  // a row's two sums by part, double-buffered by pass
  __shared__ float4 red[T][2][P * kWave];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x >> 6;
  const int team = wave / P, part = wave - team * P;
  const int C4 = C >> 2;
  const float Cf = (float)C;
  const int c4 = part * kWave + lane;
  const bool in = c4 < C4;
  const int col = in ? c4 : C4 - 1;  // past the row: a valid column, masked out of the sums, never stored
  const float4 w = ld4(weight + 4 * col);
  float4 ag = make_float4(0.f, 0.f, 0.f, 0.f), ab = ag;
  const int t0 = (blockIdx.x * T + team) * rpt;
  const int t1 = min(t0 + rpt, rows);
  const int last = t1 > t0 ? t1 - 1 : rows - 1;  // a team past the last row loads that row, uses nothing
  const int passes = (rpt + R - 1) / R;  // the same for every team: all reach every barrier
  for (int ps = 0; ps < passes; ps++) {
    const int row = t0 + ps * R;
    bool live[R];
    int rq[R];
    size_t off[R];
#pragma unroll
    for (int q = 0; q < R; q++) {
      live[q] = row + q < t1;
      rq[q] = live[q] ? row + q : last;
      off[q] = 4 * ((size_t)rq[q] * C4 + col);
    }
    float4 x[R], dy[R], dx[R], ra[kRes ? R : 1], rb[kRes ? R : 1];
    float m[R], r[R];
#pragma unroll
    for (int q = 0; q < R; q++) {
      x[q] = ld_nt4(inp + off[q]);
      dy[q] = ld_nt4(dout + off[q]);
    }
#pragma unroll
    for (int q = 0; q < R; q++) {
      m[q] = mean[rq[q]];
      r[q] = rstd[rq[q]];
    }
#pragma unroll
    for (int q = 0; q < R; q++) dx[q] = kDinp == kDinpNone ? zero4() : ld_nt4(dinp + off[q]);
    if (kRes) {
      // rdy is loaded even when it is rdx (same): a valid address, never used
#pragma unroll
      for (int q = 0; q < R; q++) {
        ra[kRes ? q : 0] = kAssign ? zero4() : ld_nt4(rdx + off[q]);
        rb[kRes ? q : 0] = kAssign ? zero4() : ld_nt4(rdy + off[q]);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    float4 xh[R], dn[R];
#pragma unroll
    for (int q = 0; q < R; q++) {
      xh[q].x = (x[q].x - m[q]) * r[q]; dn[q].x = dy[q].x * w.x;
      xh[q].y = (x[q].y - m[q]) * r[q]; dn[q].y = dy[q].y * w.y;
      xh[q].z = (x[q].z - m[q]) * r[q]; dn[q].z = dy[q].z * w.z;
      xh[q].w = (x[q].w - m[q]) * r[q]; dn[q].w = dy[q].w * w.w;
      float s1 = in ? ((dn[q].x + dn[q].y) + dn[q].z) + dn[q].w : -0.0f;
      float s2 = in ? ((dn[q].x * xh[q].x + dn[q].y * xh[q].y) + dn[q].z * xh[q].z) + dn[q].w * xh[q].w : -0.0f;
      s1 = wave_sum(s1);
      s2 = wave_sum(s2);
      if (lane == 0) {
        parts[ps & 1][team][q][part][0] = s1;
        parts[ps & 1][team][q][part][1] = s2;
      }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < R; q++) {
      if (!live[q]) break;  // the same for the team's wavefronts; dead rows are all at the end
      float s1 = parts[ps & 1][team][q][0][0], s2 = parts[ps & 1][team][q][0][1];
#pragma unroll
      for (int k = 1; k < P; k++) {
        s1 += parts[ps & 1][team][q][k][0];
        s2 += parts[ps & 1][team][q][k][1];
      }
      const float dnm = s1 / Cf, dnxm = s2 / Cf;
      float4 o;
      o.x = dx[q].x + r[q] * (dn[q].x - dnm - xh[q].x * dnxm);
      o.y = dx[q].y + r[q] * (dn[q].y - dnm - xh[q].y * dnxm);
      o.z = dx[q].z + r[q] * (dn[q].z - dnm - xh[q].z * dnxm);
      o.w = dx[q].w + r[q] * (dn[q].w - dnm - xh[q].w * dnxm);
      if (in) {
        if (kDinp == kDinpRw) {
          if (kNt)
            st_nt4(dinp + off[q], o);
          else
            st4(dinp + off[q], o);
        }
        if (kRes) {
          float4 a = add4(ra[kRes ? q : 0], o);
          if (same) {
            a = add4(a, o);
          } else {
            st_nt4(rdy + off[q], add4(rb[kRes ? q : 0], o));
          }
          st_nt4(rdx + off[q], a);
        }
      }
      ab.x += dy[q].x; ag.x += dy[q].x * xh[q].x;
      ab.y += dy[q].y; ag.y += dy[q].y * xh[q].y;
      ab.z += dy[q].z; ag.z += dy[q].z * xh[q].z;
      ab.w += dy[q].w; ag.w += dy[q].w * xh[q].w;
    }
  }
  red[team][0][c4] = ag;
  red[team][1][c4] = ab;
  __syncthreads();
  float *prow = partial + (size_t)blockIdx.x * 2 * C;
  for (int e = threadIdx.x; e < 2 * C4; e += P * T * kWave) {
    const int which = e >= C4 ? 1 : 0;
    const int cc = e - which * C4;
    float4 t = red[0][which][cc];
#pragma unroll
    for (int k = 1; k < T; k++) t = add4(t, red[k][which][cc]);
    float *q = prow + 4 * (which * C4 + cc);
    if (kTail) {
      st_dev(q, t.x); st_dev(q + 1, t.y); st_dev(q + 2, t.z); st_dev(q + 3, t.w);
    } else {
      st4(q, t);
    }
  }
  if (kTail) ln_bwd_tail<P * T * kWave>(partial, (int)gridDim.x, C, dweight, dbias);
}

// What a backward kernel whose register budget does not depend on it does with
// dinp and the residual targets: the kDinp and kAssign of k_ln_bwd_vec, the
// same in every thread.
struct LnBwdMode {
  bool read_dinp, write_dinp, assign, same;
};

// The terms of a row slot: xhat and dout * w.
__device__ __forceinline__ float4 ln_xhat4(float4 x, float m, float r) {
  return make_float4((x.x - m) * r, (x.y - m) * r, (x.z - m) * r, (x.w - m) * r);
}
__device__ __forceinline__ float4 mul4(float4 a, float4 b) {
  return make_float4(a.x * b.x, a.y * b.y, a.z * b.z, a.w * b.w);
}
// dinp + r (dn - mean(dn) - xhat mean(dn xhat))
__device__ __forceinline__ float4 ln_dinp4(float4 dx, float r, float4 dn, float4 xh, float dnm, float dnxm) {
  return make_float4(dx.x + r * (dn.x - dnm - xh.x * dnxm), dx.y + r * (dn.y - dnm - xh.y * dnxm),
                     dx.z + r * (dn.z - dnm - xh.z * dnxm), dx.w + r * (dn.w - dnm - xh.w * dnxm));
}

// A lane's share of a row's two sums.
template <int V>
__device__ __forceinline__ void ln_bwd_lane_sums(const float4 (&x)[V], const float4 (&dy)[V], const float4 (&w)[V],
                                                 float m, float r, const Cols<V, true> &cl, float &s1, float &s2) {
  s1 = s2 = 0.0f;
#pragma unroll
  for (int v = 0; v < V; v++) {
    const float4 xh = ln_xhat4(x[v], m, r), dn = mul4(dy[v], w[v]);
    s1 += cl.sel(v, 0, dn.x); s2 += cl.sel(v, 0, dn.x * xh.x);
    s1 += cl.sel(v, 1, dn.y); s2 += cl.sel(v, 1, dn.y * xh.y);
    s1 += cl.sel(v, 2, dn.z); s2 += cl.sel(v, 2, dn.z * xh.z);
    s1 += cl.sel(v, 3, dn.w); s2 += cl.sel(v, 3, dn.w * xh.w);
  }
}

// One row's outputs in a lane's slots, from its two sums over C.
template <int V, bool kRes>
__device__ __forceinline__ void ln_bwd_row_out(const float4 (&x)[V], const float4 (&dy)[V], const float4 (&w)[V],
                                               const float4 (&dx)[V], const float4 (&ra)[kRes ? V : 1],
                                               const float4 (&rb)[kRes ? V : 1], float m, float r, float dnm,
                                               float dnxm, const Cols<V, true> &cl, LnBwdMode md, float *dinp,
                                               float *rdx, float *rdy) {
#pragma unroll
  for (int v = 0; v < V; v++) {
    const float4 o = ln_dinp4(dx[v], r, mul4(dy[v], w[v]), ln_xhat4(x[v], m, r), dnm, dnxm);
    if (cl.any(v)) {
      if (md.write_dinp) cl.put(dinp, v, o);
      if (kRes) {
        float4 a = add4(ra[kRes ? v : 0], o);
        if (md.same)
          a = add4(a, o);
        else
          cl.put(rdy, v, add4(rb[kRes ? v : 0], o));
        cl.put(rdx, v, a);
      }
    }
  }
}

// Backward for rows of more than 2,048 channels: a workgroup of W wavefronts
// takes rpw consecutive rows, R at a time, V float4 of each per lane. A row's
// two sums are a lane sum, a wavefront sum and the W wavefronts' sums in order
// (one barrier per pass, LDS double-buffered by pass); dweight/dbias terms are
// added in registers in row order, and since a lane keeps its columns for all
// of the workgroup's rows, they go straight to the workgroup's partial row.
// Memory-bound: 4,092 x 4,096 in 50.9 us (5.3 TB/s), 167 us in the lane loops,
// which read x and dout three times and add a column's rows one load at a time.
// Above 4,096 channels one row at a time fits the registers, and less overlaps:
// with the column sums 2,048 x 6,144 51 us (147 in the lane loops), 2,000 x 8,192
// 64 (188).
template <int V, int W, int R, bool kRes>
__global__ __launch_bounds__(W * kWave) void k_ln_bwd_wide(float *__restrict__ dinp, float *__restrict__ partial,
                                                           const float *__restrict__ dout,
                                                           const float *__restrict__ inp,
                                                           const float *__restrict__ weight,
                                                           const float *__restrict__ mean,
                                                           const float *__restrict__ rstd, int rows, int C, int rpw,
                                                           float *__restrict__ rdx, float *__restrict__ rdy,
                                                           LnBwdMode md) {
  __shared__ float part[2][R][W][2];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & (kWave - 1);
  const float Cf = (float)C;
  const Cols<V, true> cl(threadIdx.x, W * kWave, C);
  float4 w[V], ag[V], ab[V];
#pragma unroll
  for (int v = 0; v < V; v++) {
    w[v] = ld4(weight + cl.at[v]);
    ag[v] = ab[v] = zero4();
  }
  const int row0 = blockIdx.x * rpw, row1 = min(row0 + rpw, rows);
  for (int row = row0, ps = 0; row < row1; row += R, ps ^= 1) {
    float4 x[R][V], dy[R][V], dx[R][V], ra[R][kRes ? V : 1], rb[R][kRes ? V : 1];
    float m[R], r[R];
    size_t off[R];
#pragma unroll
    for (int q = 0; q < R; q++) {  // rows past the end repeat the last one: computed, neither stored nor summed
      const int rq = min(row + q, row1 - 1);
      off[q] = (size_t)rq * C;
      m[q] = mean[rq];
      r[q] = rstd[rq];
#pragma unroll
      for (int v = 0; v < V; v++) {
        x[q][v] = ld_nt4(inp + off[q] + cl.at[v]);
        dy[q][v] = ld_nt4(dout + off[q] + cl.at[v]);
      }
    }
#pragma unroll
    for (int q = 0; q < R; q++)
#pragma unroll
      for (int v = 0; v < V; v++) {
        dx[q][v] = md.read_dinp ? ld_nt4(dinp + off[q] + cl.at[v]) : zero4();
        if (kRes) {
          ra[q][kRes ? v : 0] = md.assign ? zero4() : ld_nt4(rdx + off[q] + cl.at[v]);
          rb[q][kRes ? v : 0] = md.assign ? zero4() : ld_nt4(rdy + off[q] + cl.at[v]);
        }
      }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < R; q++) {
      float s1, s2;
      ln_bwd_lane_sums<V>(x[q], dy[q], w, m[q], r[q], cl, s1, s2);
      s1 = wave_sum(s1);
      s2 = wave_sum(s2);
      if (lane == 0) {
        part[ps][q][wave][0] = s1;
        part[ps][q][wave][1] = s2;
      }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < R; q++) {
      if (row + q >= row1) break;  // the same in every thread
      float s1 = part[ps][q][0][0], s2 = part[ps][q][0][1];
#pragma unroll
      for (int k = 1; k < W; k++) {
        s1 += part[ps][q][k][0];
        s2 += part[ps][q][k][1];
      }
      ln_bwd_row_out<V, kRes>(x[q], dy[q], w, dx[q], ra[q], rb[q], m[q], r[q], s1 / Cf, s2 / Cf, cl, md,
                              dinp + off[q], rdx + off[q], rdy + off[q]);
#pragma unroll
      for (int v = 0; v < V; v++) {
        ab[v] = add4(ab[v], dy[q][v]);
        ag[v] = add4(ag[v], mul4(dy[q][v], ln_xhat4(x[q][v], m[q], r[q])));
      }
    }
  }
  float *prow = partial + (size_t)blockIdx.x * 2 * C;
#pragma unroll
  for (int v = 0; v < V; v++)
    if (cl.any(v)) {
      cl.put(prow, v, ag[v]);
      cl.put(prow + C, v, ab[v]);
    }
}

// Backward of few rows without partial rows. What bounds it is latency: a
// launch, one round trip to memory, the reductions. A call's first workgroups
// sum dweight and dbias by themselves, 16 columns each, reading x and dout
// once more (they are in the caches): 64 groups of consecutive rows, each
// added in row order, every eighth group together, then those eight sums as a
// tree, then onto the arrays' values, or (add false) as the call's only partial
// row. The others write dinp (and the residual targets), P wavefronts per row,
// every row's loads in flight at once. The step driver's calls leave the columns
// out (ncol = 0) where nothing but its own kernels runs before its end, and one
// launch there takes them for all its LayerNorms (k_ln_small_cols_batch: 154
// against 175 us for a step of 13 LayerNorms of 256 x 384); with dense
// callbacks, which may write to the gradients again, each call sums its own, as
// a partial row. Per call, captured and cold, against the two launches of the
// larger shapes' kernels: 256 x 384 3.8 against 7.6 us, 512 x 768 6.4 against
// 10.3, 640 x 384 4.9 against 8.2. With more rows the few column workgroups
// stream too much each (8 or 32 columns a workgroup, and longer batches, moved
// that by 2 us at most), hence small_path.
constexpr int kSmallCols = 16, kSmallSlots = kSmallCols / 4, kSmallGroups = kBlock / kSmallSlots, kSmallBatch = 4;

__device__ __forceinline__ void ln_small_cols(float (*red)[2][kSmallCols], int blk, float *__restrict__ dweight,
                                              float *__restrict__ dbias, const float *__restrict__ dout,
                                              const float *__restrict__ inp, const float *__restrict__ mean,
                                              const float *__restrict__ rstd, int rows, int C, bool add) {
  const int l = threadIdx.x % kSmallSlots, g = threadIdx.x / kSmallSlots;
  const Cols<1, true> cl(blk * kSmallSlots + l, 0, C);
  // the adder thread's column: component col % 4 of slot col / 4, if that is the slot's own
  const int which = (int)threadIdx.x / kSmallCols, col = (int)threadIdx.x % kSmallCols;
  const Cols<1, true> cc(blk * kSmallSlots + col / 4, 0, C);
  const bool adder = (int)threadIdx.x < 2 * kSmallCols && cc.own(0, col & 3);
  float *const dst = (which ? dbias : dweight) + cc.at[0] + (col & 3);
  const float prev = adder && add ? *dst : -0.0f;
  float4 ag = zero4(), ab = zero4();
  const int J = (rows + kSmallGroups - 1) / kSmallGroups;
  const int j0 = min(g * J, rows), j1 = min(j0 + J, rows);
  for (int b = j0; b < j1; b += kSmallBatch) {
    float4 x[kSmallBatch], dy[kSmallBatch];
    float m[kSmallBatch], r[kSmallBatch];
#pragma unroll
    for (int q = 0; q < kSmallBatch; q++) {
      const int row = min(b + q, j1 - 1);
      x[q] = ld4(inp + (size_t)row * C + cl.at[0]);
      dy[q] = ld4(dout + (size_t)row * C + cl.at[0]);
      m[q] = mean[row];
      r[q] = rstd[row];
    }
#pragma unroll
    for (int q = 0; q < kSmallBatch; q++) {
      if (b + q >= j1) break;
      ab = add4(ab, dy[q]);
      ag = add4(ag, mul4(dy[q], ln_xhat4(x[q], m[q], r[q])));
    }
  }
  *reinterpret_cast<float4 *>(&red[g][0][4 * l]) = ag;
  *reinterpret_cast<float4 *>(&red[g][1][4 * l]) = ab;
  __syncthreads();
  if (adder) {
    float t[8];
#pragma unroll
    for (int k = 0; k < 8; k++) {
      t[k] = red[k][which][col];
#pragma unroll
      for (int j = k + 8; j < kSmallGroups; j += 8) t[k] += red[j][which][col];
    }
    *dst = prev + (((t[0] + t[1]) + (t[2] + t[3])) + ((t[4] + t[5]) + (t[6] + t[7])));
  }
}

template <int V, int P, bool kRes>
__global__ __launch_bounds__(kBlock) void k_ln_bwd_small(float *__restrict__ dinp, float *__restrict__ dweight,
                                                         float *__restrict__ dbias, const float *__restrict__ dout,
                                                         const float *__restrict__ inp,
                                                         const float *__restrict__ weight,
                                                         const float *__restrict__ mean,
                                                         const float *__restrict__ rstd, int rows, int C, int ncol,
                                                         int add, float *__restrict__ rdx, float *__restrict__ rdy,
                                                         LnBwdMode md) {
  __shared__ __align__(16) float red[kSmallGroups][2][kSmallCols];
  if ((int)blockIdx.x < ncol) {
    ln_small_cols(red, blockIdx.x, dweight, dbias, dout, inp, mean, rstd, rows, C, add != 0);
    return;
  }
  constexpr int T = kWavesPerBlock / P;  // rows per workgroup
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & (kWave - 1);
  const int row = ((int)blockIdx.x - ncol) * T + wave / P;
  if (P == 1 && row >= rows) return;  // P > 1: one row per workgroup, all of them rows
  const Cols<V, true> cl(wave % P * kWave + lane, P * kWave, C);
  const size_t off = (size_t)row * C;
  const float m = mean[row], r = rstd[row];
  float4 x[V], dy[V], w[V], dx[V], ra[kRes ? V : 1], rb[kRes ? V : 1];
#pragma unroll
  for (int v = 0; v < V; v++) {
    x[v] = ld_nt4(inp + off + cl.at[v]);
    dy[v] = ld_nt4(dout + off + cl.at[v]);
    w[v] = ld4(weight + cl.at[v]);
    dx[v] = md.read_dinp ? ld_nt4(dinp + off + cl.at[v]) : zero4();
    if (kRes) {
      ra[kRes ? v : 0] = md.assign ? zero4() : ld_nt4(rdx + off + cl.at[v]);
      rb[kRes ? v : 0] = md.assign ? zero4() : ld_nt4(rdy + off + cl.at[v]);
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  float s1, s2;
  ln_bwd_lane_sums<V>(x, dy, w, m, r, cl, s1, s2);
  s1 = wave_sum(s1);
  s2 = wave_sum(s2);
  if (P > 1) {
    float(*part)[2] = reinterpret_cast<float(*)[2]>(&red[0][0][0]);
    if (lane == 0) {
      part[wave][0] = s1;
      part[wave][1] = s2;
    }
    __syncthreads();
    s1 = part[0][0];
    s2 = part[0][1];
#pragma unroll
    for (int k = 1; k < P; k++) {
      s1 += part[k][0];
      s2 += part[k][1];
    }
  }
  ln_bwd_row_out<V, kRes>(x, dy, w, dx, ra, rb, m, r, s1 / (float)C, s2 / (float)C, cl, md, dinp + off, rdx + off,
                          rdy + off);
}

// Backward for the rows that no kernel above takes (C < 4 or beyond 8,192): one
// wavefront per row writes dinp, and thread-per-channel column sums over the
// workgroup's rows. Both read dout and inp from memory, the sums what the rows
// have left in the cache (50 x 8,200 86 us, 90 with the sums first); where dinp
// is one of them (in_place) the sums come first, since a row's terms are those
// of the arrays as they were.
template <bool kColsFirst>
__global__ __launch_bounds__(kBlock) void k_ln_bwd_scalar(float *dinp, float *partial, const float *dout,
                                                          const float *inp, const float *weight,
                                                          const float *mean, const float *rstd, int rows,
                                                          int C, int rpb) {
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x >> 6;
  const float Cf = (float)C;
  const int row0 = blockIdx.x * rpb;
  const int row1 = min(row0 + rpb, rows);
  const auto write_rows = [&] {
    for (int row = row0 + wave; row < row1; row += kWavesPerBlock) {
      const float *x = inp + (size_t)row * C;
      const float *dy = dout + (size_t)row * C;
      float *dx = dinp + (size_t)row * C;
      const float m = mean[row], r = rstd[row];
      float s1 = 0.0f, s2 = 0.0f;
      for (int c = lane; c < C; c += kWave) {
        const float xhat = (x[c] - m) * r;
        const float dnorm = dy[c] * weight[c];
        s1 += dnorm;
        s2 += dnorm * xhat;
      }
      s1 = wave_sum(s1);
      s2 = wave_sum(s2);
      const float dnm = s1 / Cf, dnxm = s2 / Cf;
      for (int c = lane; c < C; c += kWave) {
        const float xhat = (x[c] - m) * r;
        const float dnorm = dy[c] * weight[c];
        dx[c] += r * (dnorm - dnm - xhat * dnxm);
      }
    }
  };
  if (!kColsFirst) write_rows();
  float *prow = partial + (size_t)blockIdx.x * 2 * C;
  for (int c = threadIdx.x; c < C; c += kBlock) {
    float g = 0.0f, b = 0.0f;
    for (int row = row0; row < row1; row++) {
      const float dy = dout[(size_t)row * C + c];
      const float xhat = (inp[(size_t)row * C + c] - mean[row]) * rstd[row];
      b += dy;
      g += dy * xhat;
    }
    prow[c] = g;
    prow[C + c] = b;
  }
  if (kColsFirst) {
    __syncthreads();
    write_rows();
  }
}

// Column totals of the partial rows, added to dweight (columns [0,C)) and
// dbias (columns [C,2C)). Workgroup: 32 columns x 16 groups; group k sums the
// partial rows [k*J, (k+1)*J), J = ceil(nblk/16) <= 64 (RowChains), 32
// loads in flight per batch; the 16 group sums are then added in group order.
// 32 columns rather than 64 spread one LayerNorm's totals over twice the
// workgroups (48 at C = 768): the per-op backward at 8,192 x 768 took 22.3-22.6
// against 23.3 us cold, and the step's batched launch 12.7 against 13.1-13.3 us
// (16 columns: 22.6 us). The order of the additions does not depend on it.
constexpr int kRedGroups = 16;
constexpr int kRedCols = 32;
static_assert(kRedGroups == kTailGroups, "the in-launch column sums follow the column-sum kernel's order");
constexpr int kRedBatch = 32;
static_assert(kMaxPartialRows <= kRedGroups * 2 * kRedBatch, "two load batches per group at most");
__device__ __forceinline__ void ln_bwd_reduce_tile(float *dweight, float *dbias, const float *partial, int nblk,
                                                   int C, float (*red)[kRedCols]) {
  const int cl = threadIdx.x % kRedCols;
  const int g = threadIdx.x / kRedCols;
  const int col = blockIdx.x * kRedCols + cl;
  const int C2 = 2 * C;
  const int J = (nblk + kRedGroups - 1) / kRedGroups;
  const int j0 = g * J, j1 = min(j0 + J, nblk);
  const int cc = col < C2 ? col : C2 - 1;
  // the value the total is added to, loaded with the partial rows rather than
  // after them (one memory round trip fewer at the end)
  float* const dst = col < C ? dweight + col : dbias + (cc - C);
  const float prev = g == 0 && col < C2 ? *dst : 0.0f;
  RowChains acc;
  for (int b = j0; b < j1; b += kRedBatch) {
    float v[kRedBatch];
#pragma unroll
    for (int q = 0; q < kRedBatch; q++) v[q] = partial[(size_t)min(b + q, j1 - 1) * C2 + cc];
    acc.add(v, j1 - b);
  }
  red[g][cl] = acc.sum();
  __syncthreads();
  if (g == 0 && col < C2) {
    float t = red[0][cl];
#pragma unroll
    for (int k = 1; k < kRedGroups; k++) t += red[k][cl];
    *dst = prev + t;
  }
}

// Several LayerNorm backwards' column totals in one launch (blockIdx.y picks
// the job).
constexpr int kMaxReduceJobs = 32;
struct LnReduceBatch {
  LnReduceJob job[kMaxReduceJobs];
};
__global__ __launch_bounds__(kRedCols * kRedGroups) void k_ln_bwd_reduce_batch(LnReduceBatch b, int C) {
  __shared__ float red[kRedGroups][kRedCols];
  const LnReduceJob &j = b.job[blockIdx.y];
  ln_bwd_reduce_tile(j.dweight, j.dbias, j.partial, j.nblk, C, red);
}

// The columns of several few-row LayerNorms in one launch (blockIdx.y picks the job).
__global__ __launch_bounds__(kBlock) void k_ln_small_cols_batch(LnReduceBatch b, int rows, int C) {
  __shared__ __align__(16) float red[kSmallGroups][2][kSmallCols];
  const LnReduceJob &j = b.job[blockIdx.y];
  ln_small_cols(red, blockIdx.x, j.dweight, j.dbias, j.dout, j.inp, j.mean, j.rstd, rows, C, true);
}

// Which kernels take rows of C channels, at any alignment: one wavefront per
// row up to 2,048, a workgroup per row up to 8,192, else the lane loops.
bool row_in_wave(int C) { return C >= 4 && C <= kMaxV * kWave * 4; }
bool row_in_block(int C) { return C > kMaxV * kWave * 4 && C <= kMaxWide; }
int slots_of(int C, int lanes) { return ((C + 3) / 4 + lanes - 1) / lanes; }  // float4 per lane

// Scalar path: workgroups of 4 wavefronts, at most max_blocks of them.
void bwd_shape(int rows, int max_blocks, int *nblk, int *rpb) {
  int nb = (rows + kWavesPerBlock - 1) / kWavesPerBlock;
  if (nb > max_blocks) nb = max_blocks;
  if (nb < 1) nb = 1;
  int per = (rows + nb - 1) / nb;
  per = (per + kWavesPerBlock - 1) / kWavesPerBlock * kWavesPerBlock;
  *rpb = per;
  *nblk = (rows + per - 1) / per;
}

// Vector path shapes: 8 wavefronts per workgroup, 4 when a lane holds more
// than 4 float4 of a row. Each wavefront takes S consecutive rows (S = 2 while
// C <= 768, else 1) while that leaves at most max_blocks workgroups, else
// more: at 16,384 x 768 one pass over 1,024 workgroups took 72 us for the
// fused pair against 81 us with two passes over 512. The plain backward and
// the fused pair share this shape (the rows of each wavefront and workgroup),
// hence the order in which dweight/dbias are summed, so that the pair is
// bit-identical to the plain backward followed by residual_backward.
// Rows in flight differ: the fused pair loads both of its rows at once (214
// registers, two wavefronts per SIMD); the plain backward takes one row at a
// time within 128 registers, four wavefronts per SIMD, which measured 18.9
// against 20.1 us at 8,192 x 768 (35.9 against 39.5 us at 16,384) with the
// same sums.
struct BwdCfg {
  int W, S, R, MINW;
};
constexpr BwdCfg bwd_cfg(int V, bool res) {
  return BwdCfg{V <= 4 ? 8 : 4, V <= 3 ? 2 : 1, (V <= 3 && res) ? 2 : 1, (V <= 3 && !res) ? 4 : 1};
}
void bwd_shape_vec(int rows, BwdCfg k, int max_blocks, int *nblk, int *rpw) {
  const int per_wave = (rows + max_blocks * k.W - 1) / (max_blocks * k.W);
  *rpw = per_wave < k.S ? k.S : per_wave;
  *nblk = (rows + k.W * *rpw - 1) / (k.W * *rpw);
}

// Compute units of the current device (cached per device; 256 if unknown).
int cu_count() {
  static int cus[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) {
    (void)hipGetLastError();  // leave no error for the next launch check to report
    return 256;
  }
  if (cus[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) {
      (void)hipGetLastError();
      n = 256;
    }
    cus[dev] = n;
  }
  return cus[dev];
}

// Team path, V = 3 (C/4 in 129..192), while the rows fill the GPU at most
// once at 32 rows per CU (8,192 on MI355X): teams of 3 wavefronts, 4 teams
// per workgroup, at least 4 rows per team (16 per workgroup, 512 workgroups
// at 8,192 rows), more while that would leave more than max_blocks
// workgroups. The plain backward keeps 2 rows in flight (70 registers), the
// fused pair 4 (156). Beyond that the two-rows-per-wavefront kernels are
// used: at 16,384 x 768 they measured as fast for the fused pair and faster
// for the plain backward (41.7 against 45.0 us with the column sums).
constexpr int kTeamParts = 3, kTeams = 4, kTeamRows = 4;
bool team_path(int rows, int C) {
  return (C & 3) == 0 && slots_of(C, kWave) == kTeamParts && rows <= cu_count() * 32;
}
void team_shape(int rows, int max_blocks, int *nblk, int *rpt) {
  const int per_team = (rows + max_blocks * kTeams - 1) / (max_blocks * kTeams);
  *rpt = per_team < kTeamRows ? kTeamRows : per_team;
  *nblk = (rows + kTeams * *rpt - 1) / (kTeams * *rpt);
}

// Workgroups (partial rows) of a vector-path call, for sizing its workspace:
// at V = 3 the larger of the two kernels' counts, so that the size does not
// depend on the device the call later runs on.
int vec_blocks(int rows, int C, bool res, int max_blocks) {
  int nblk, rpw;
  const int V = slots_of(C, kWave);
  bwd_shape_vec(rows, bwd_cfg(V, res), max_blocks, &nblk, &rpw);
  if (V == kTeamParts) {
    int nt, rpt;
    team_shape(rows, max_blocks, &nt, &rpt);
    if (nt > nblk) nblk = nt;
  }
  return nblk;
}

// Workgroup-per-row path: W wavefronts per workgroup, at least 4 rows each (as
// many partial rows as the scalar path may take, which sizes the workspace),
// at most 512 workgroups.
constexpr int kWideWaves = 8, kWideRows = 4;
void wide_shape(int rows, int max_blocks, int *nblk, int *rpw) {
  const int cap = std::min(max_blocks, kMaxScalarBlocks);
  const int per = (rows + cap - 1) / cap;
  *rpw = per < kWideRows ? kWideRows : per;
  *nblk = (rows + *rpw - 1) / *rpw;
}

// The backward without partial rows (k_ln_bwd_small). The lines are where it
// meets the two launches, captured and cold, the plain backward and the pair:
//   up to 512 rows      of 1,024 channels 8.3 against 8.3 and 9.6 against 10.3
//                       us, 768 6.4 against 10.3, but 1,280 8.8 against 8.3;
//                       beyond 1,536 the two launches are slower again: 2,048
//                       9.1 against 10.2, 256 x 4,096 7.8 against 11.9;
//   up to 1,024, cols'  1,024 x 256 6.6 against 7.5, 640 x 384 4.9 against
//   arrays aligned      8.2, but 1,024 x 320 10.8 against 8.3, 896 x 320 8.5
//                       against 8.3;
//   the same, at other  768 x 256 6.4 against 7.5 and 9.4 against 8.1, but
//   addresses or widths 896 x 256 10.7 against 7.6, 640 x 384 9.0 against 8.4
//                       (the column workgroups' 64 bytes of a row then lie in
//                       two lines as often as not).
bool small_path(int rows, int C, const float *dout, const float *inp) {
  if (!row_in_wave(C) && !row_in_block(C)) return false;
  const size_t n = (size_t)rows * C;
  if (rows <= 512) return n <= ((size_t)1 << 19) || (C > 1536 && n <= ((size_t)1 << 20));
  const bool aligned = (C & 3) == 0 && aligned16(dout) && aligned16(inp);
  return rows <= 1024 && n <= (size_t)(aligned ? 4 : 3) << 16;
}

// Rows per wavefront of the fused forward: two while one wavefront per row
// would fill the GPU only once (the reads and writes of a single round of
// wavefronts cannot overlap; measured 17.7 against 18.8 us at 8,192 x 768),
// else one (35.0 against 37.1 us at 16,384 x 768), and one again while a SIMD
// waits for its rows anyway (fwd_early), where a wavefront's second row only
// adds to the latency (1,024 x 768 4.6 against 5.4 us, 256 x 384 3.3 against
// 3.9, 512 x 1,600 5.7 against 7.9). The plain forward keeps one (9.3 against
// 9.6 us with two at 8,192 x 768).
// Weight and bias loaded early (ln_row_out): up to two rows per SIMD, of rows
// that keep it waiting (2,048 x 768 6.4 against 6.9 us, but 2,048 x 1,600 12.1
// against 11.0 and 2,000 x 1,024 8.1 against 7.8).
bool fwd_early(int rows, int C) { return rows <= cu_count() * 8 && (size_t)rows * C <= ((size_t)3 << 19); }
int fwd_rpw(int rows, int C, bool res) {
  if (!res) return 1;
  return !fwd_early(rows, C) && rows <= cu_count() * 32 ? 2 : 1;
}

}  // namespace

int layernorm_backward_blocks(int rows, int C, bool res, int max_blocks) {
  if (rows <= 0) return 0;
  if (row_in_wave(C)) return vec_blocks(rows, C, res, max_blocks);
  int nblk, rpb;
  if (row_in_block(C)) {
    wide_shape(rows, max_blocks, &nblk, &rpb);
    return nblk;
  }
  bwd_shape(rows, max_blocks < kMaxScalarBlocks ? max_blocks : kMaxScalarBlocks, &nblk, &rpb);
  return nblk;
}

// An upper bound on the partial rows of every call with at most `rows` rows
// and at most C channels, on any path. A path's count is not monotone in the
// rows (once a call would exceed the cap, each workgroup takes more rows and
// the count drops below the cap), but it never exceeds
// min(cap, ceil(rows / floor)), where floor is the fewest rows a workgroup of
// that path takes: 4 on the scalar path (cap 512) and on the wave-per-row path
// above 1,024 channels (one row per wavefront, four wavefronts), 8 from 772
// channels (eight wavefronts, one row each), 16 below (eight wavefronts of two
// rows, or four teams of four rows; cap 1,024). Sizing a workspace by this
// bound at a config's rows therefore covers every smaller call.
int layernorm_backward_blocks_bound(int rows, int C) {
  const auto cap_div = [rows](int cap, int floor) {
    const long long q = ((long long)rows + floor - 1) / floor;
    return (int)(q < cap ? q : cap);
  };
  int nb = cap_div(kMaxScalarBlocks, 4);
  if (C > kWave * 4 * 4) nb = std::max(nb, cap_div(kMaxPartialRows, 4));
  if (C > kWave * 4 * 3) nb = std::max(nb, cap_div(kMaxPartialRows, 8));
  nb = std::max(nb, cap_div(kMaxPartialRows, 16));
  return rows > 0 ? nb : 0;
}

size_t layernorm_backward_scratch(int rows, int C) {
  return (size_t)layernorm_backward_blocks_bound(rows, C) * 2 * (size_t)C * sizeof(float);
}

namespace {
// Rows of 4 to 8,192 channels, at any alignment.
template <bool kRes>
void launch_ln_fwd_rows(float *out, float *mean, float *rstd, const float *inp, const float *weight,
                        const float *bias, int rows, int C, float *res, const float *inp2) {
  if (row_in_block(C)) {
    // 4 wavefronts with 3 or 4 float4 per lane up to 4,096 channels, 8 up to 8,192
    const bool w8 = C > 4 * kWave * 4 * 4;
    const int V = slots_of(C, (w8 ? 8 : 4) * kWave);
    const auto go = [&](auto k, int W) {
      launch(k, dim3(rows), dim3(W * kWave), 0, out, mean, rstd, inp, weight, bias, C, res, inp2);
    };
    if (!w8 && V <= 3) go(k_ln_fwd_wide<3, 4, kRes>, 4);
    else if (!w8) go(k_ln_fwd_wide<4, 4, kRes>, 4);
    else if (V <= 3) go(k_ln_fwd_wide<3, 8, kRes>, 8);
    else go(k_ln_fwd_wide<4, 8, kRes>, 8);
    return;
  }
  const bool rag = (C & 3) != 0, early = fwd_early(rows, C);
  const int rpw = rag ? 1 : fwd_rpw(rows, C, kRes);
  const dim3 grid(grid_for((size_t)rows, (size_t)kWavesPerBlock * rpw)), block(kBlock);
  const auto go = [&](auto k) { launch(k, grid, block, 0, out, mean, rstd, inp, weight, bias, rows, C, res, inp2); };
  switch (slots_of(C, kWave)) {
#define UGK_LN_FWD(v)                                                  \
  case v:                                                              \
    if (rag && early) go(k_ln_fwd_vec<v, kRes, 1, true, true>);        \
    else if (rag) go(k_ln_fwd_vec<v, kRes, 1, true, false>);           \
    else if (early) go(k_ln_fwd_vec<v, kRes, 1, false, true>);         \
    else if (rpw == 1) go(k_ln_fwd_vec<v, kRes, 1, false, false>);     \
    else go(k_ln_fwd_vec<v, kRes, 2, false, false>);                   \
    break;
    UGK_LN_FWD(1) UGK_LN_FWD(2) UGK_LN_FWD(3) UGK_LN_FWD(4)
    UGK_LN_FWD(5) UGK_LN_FWD(6) UGK_LN_FWD(7) UGK_LN_FWD(8)
#undef UGK_LN_FWD
  }
}
}  // namespace

int launch_residual_layernorm_forward(float *res, float *out, float *mean, float *rstd, const float *x,
                                      const float *y, const float *weight, const float *bias, int rows,
                                      int C) {
  if (rows == 0) return 0;
  if (layernorm_exact() || !(row_in_wave(C) || row_in_block(C))) {
    if (int e = launch_residual_forward(res, x, y, (size_t)rows * C)) return e;
    return launch_layernorm_forward(out, mean, rstd, res, weight, bias, rows, C);
  }
  launch_ln_fwd_rows<true>(out, mean, rstd, x, weight, bias, rows, C, res, y);
  return check_launch("residual_layernorm_forward");
}

int launch_encoder_layernorm_forward(float *enc, float *out, float *mean, float *rstd, int *inp,
                                     const float *wte, const float *wpe, const float *weight, const float *bias,
                                     int B, int T, int C, const IdCheck &ids) {
  const int rows = B * T;
  if (rows == 0) return 0;
  if (layernorm_exact() || !row_in_wave(C) || (C & 3) != 0) {
    if (int e = launch_encoder_forward(enc, inp, wte, wpe, B, T, C, ids)) return e;
    return launch_layernorm_forward(out, mean, rstd, enc, weight, bias, rows, C);
  }
  const int V = slots_of(C, kWave);
  const int rpw = fwd_rpw(rows, C, true);
  const dim3 grid(grid_for((size_t)rows, (size_t)kWavesPerBlock * rpw)), block(kBlock);
  const auto go = [&](auto k) {
    launch(k, grid, block, 0, enc, out, mean, rstd, inp, ids, wte, wpe, weight, bias, rows, T, C);
  };
  switch (V) {
#define UGK_ENC_LN(v)                                             \
  case v:                                                         \
    if (fwd_early(rows, C)) go(k_enc_ln_fwd_vec<v, 1, true>);        \
    else if (rpw == 1) go(k_enc_ln_fwd_vec<v, 1, false>);         \
    else go(k_enc_ln_fwd_vec<v, 2, false>);                       \
    break;
    UGK_ENC_LN(1) UGK_ENC_LN(2) UGK_ENC_LN(3) UGK_ENC_LN(4)
    UGK_ENC_LN(5) UGK_ENC_LN(6) UGK_ENC_LN(7) UGK_ENC_LN(8)
#undef UGK_ENC_LN
  }
  return check_launch("encoder_layernorm_forward");
}

namespace {
// ---- exact mode: train_bnn.c's order of every addition ------------------------
// train_bnn.c:81-115 and :439-477 add each row's terms one column at a time
// (c = 0, 1, ..., C-1), and dweight/dbias one row at a time. The exact kernels
// keep those orders, each sum a serial chain in one lane of wavefront 0, which
// does nothing but the chains' additions; fifteen loader wavefronts keep it fed:
//   rows: a workgroup per 60 rows. The loaders stream 64-column tiles of the
//     rows, three tiles ahead in registers, and stage each row's terms in LDS
//     (the forward: x, then (x - mean)^2; the backward: dout * w and
//     dout * w * xhat), row-major at a pitch of 68 floats, so that the chains
//     read four terms at a time without bank conflicts. One chain per row
//     (lane = row; lanes 60-63 follow copies and store nothing; 60 rows make a
//     tile whole loader slots, scalar and float4). Then every wavefront writes out (or adds to dinp) whole
//     rows with the row statistics.
//   columns: a workgroup per 16 columns. The loaders stage 240-row tiles of
//     the dweight terms dout * xhat and the dbias terms dout, transposed (a
//     column's terms contiguous, pitch 244 floats); lanes 0-15 chain dweight,
//     lanes 16-31 dbias, one row after another, from the values the arrays hold.
// Every term is rounded as the CPU rounds it (no product is contracted into an
// fma; the square root and quotients are IEEE's), so every result is
// train_bnn.c's bit for bit. The backward's row and column workgroups are
// independent and share one launch. kVec: C a multiple of 4 and the row
// arrays 16-byte aligned, every global access of the rows a float4 (a quarter
// of the memory instructions, which bound these kernels); otherwise scalar
// accesses, any C, any alignment.
constexpr int kExLoaders = 15;
constexpr int kExThreads = (kExLoaders + 1) * kWave;
constexpr int kExLoadLanes = kExLoaders * kWave;
constexpr int kExDepth = 3;  // tiles in registers ahead of the chains
constexpr int kExRows = 60;  // rows per row workgroup (one chain per lane of wavefront 0)
constexpr int kExTile = 64;  // columns per tile of a row workgroup
constexpr int kExPitch = kExTile + 4;
constexpr int kExSlots = (kExRows * kExTile + kExLoadLanes - 1) / kExLoadLanes;
constexpr int kExVecSlots = (kExRows * kExTile / 4 + kExLoadLanes - 1) / kExLoadLanes;
constexpr int kExApply = 8;       // scalar elements per lane in flight when the rows are written
constexpr int kExApplyVec = 4;    // float4 per lane in flight when the rows are written
constexpr int kExCols = 16;       // columns per column workgroup (two chains each)
constexpr int kExChains = 2 * kExCols;
constexpr int kExColRows = 240;   // rows per tile of a column workgroup
constexpr int kExColPitch = kExColRows + 4;
constexpr int kExColSlots = kExColRows * kExCols / kExLoadLanes;
// float4 reads per chain and batch (two batches in flight): 32 additions a
// batch in the row chains; 24 in the column chains, whose loaders hold more
// registers
constexpr int kExBatch = 8;
constexpr int kExColBatch = 6;
static_assert(kExRows <= kWave && kWave % kExCols == 0 && kExChains <= kWave, "chains in wavefront 0");
static_assert(kExRows * kExTile == kExSlots * kExLoadLanes && kExRows * kExTile / 4 == kExVecSlots * kExLoadLanes,
              "a row tile is whole loader slots, scalar and float4");
static_assert(kExColRows * kExCols == kExColSlots * kExLoadLanes && kExColRows * kExCols / 4 == kExLoadLanes,
              "a column tile is whole loader slots, scalar and float4");
static_assert(kExTile % (8 * kExBatch) == 0 && kExColRows % (8 * kExColBatch) == 0, "whole batch pairs per tile");
static_assert(kExLoadLanes % (kExTile / 4) == 0, "a loader lane keeps its float4 column in every slot");
// LDS of a row workgroup (floats): term tiles (a row per lane of wavefront 0),
// per-row statistics and sums
constexpr int ex_row_lds(int arrays) { return 2 * arrays * kWave * kExPitch + 4 * kWave; }
constexpr int kExColLds = 2 * kExChains * kExColPitch;
constexpr int kExBwdLds = ex_row_lds(2) > kExColLds ? ex_row_lds(2) : kExColLds;

__device__ __forceinline__ float f4_get(const float4 &v, int j) {
  return j == 0 ? v.x : j == 1 ? v.y : j == 2 ? v.z : v.w;
}

template <bool kBwd, bool kVec>
__device__ __forceinline__ void ln_rows_exact(float *lds, int blk, float *__restrict__ outp, float *__restrict__ mean,
                                              float *__restrict__ rstd, const float *__restrict__ inp,
                                              const float *__restrict__ dout, const float *__restrict__ weight,
                                              const float *__restrict__ bias, int rows, int C) {
  constexpr int kArr = kBwd ? 2 : 1;  // staged term arrays
  constexpr int kTileF = kWave * kExPitch;
  constexpr int kSlots = kVec ? kExVecSlots : kExSlots;
  constexpr int kW = kVec ? 4 : 1;  // floats per lane and slot
  float *const tile = lds;  // [2][kArr][kTileF]
  float2 *const stat = reinterpret_cast<float2 *>(lds + 2 * kArr * kTileF);  // [kWave]: mean, rstd
  float2 *const rsum = stat + kWave;  // [kWave]: the backward's row sums / C
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & (kWave - 1);
  const int r0 = blk * kExRows;
  const int nt = (C + kExTile - 1) / kExTile;
  const int nu = (kBwd ? 1 : 2) * nt;  // tiles streamed: the forward reads every tile twice
  const float Cf = (float)C;
  float s[kArr];  // the chains of wavefront 0's lane: row r0 + lane
#pragma unroll
  for (int a = 0; a < kArr; a++) s[a] = 0.0f;
  if (kBwd) {
    // the rows' statistics, for the loaders' terms and the writes
    if (wave == 0) {
      const int crow = min(r0 + lane, rows - 1);
      stat[lane] = make_float2(mean[crow], rstd[crow]);
    }
    __syncthreads();
  }
  // Loader lane L = 64 lw + lane. Scalar: slot sl holds tile row lw + 15 sl,
  // column lane. float4: slot sl holds float4 f = L + 960 sl of the tile (row
  // f / 16, columns 4 (f % 16) + 0..3), the column the same in every slot.
  const int lw = wave - 1;
  const int L = lw * kWave + lane;
  float reg[kExDepth][kArr][kSlots][kW];
  float wreg[kExDepth][kW];
  auto slot_row = [&](int sl) { return kVec ? (L + kExLoadLanes * sl) / (kExTile / 4) : lw + kExLoaders * sl; };
  const int lcol = kVec ? 4 * (L % (kExTile / 4)) : lane;
  auto load_tile = [&](int u, int k) {
    const int col = min((u % nt) * kExTile + lcol, C - kW);
#pragma unroll
    for (int sl = 0; sl < kSlots; sl++) {
      const int ri = min(slot_row(sl), kExRows - 1);
      const size_t off = (size_t)min(r0 + ri, rows - 1) * C + col;
      if constexpr (kVec) {
        const float4 x = *reinterpret_cast<const float4 *>(inp + off);
        reg[k][0][sl][0] = x.x, reg[k][0][sl][1] = x.y, reg[k][0][sl][2] = x.z, reg[k][0][sl][3] = x.w;
        if (kBwd) {
          const float4 y = *reinterpret_cast<const float4 *>(dout + off);
          reg[k][kArr - 1][sl][0] = y.x, reg[k][kArr - 1][sl][1] = y.y;
          reg[k][kArr - 1][sl][2] = y.z, reg[k][kArr - 1][sl][3] = y.w;
        }
      } else {
        reg[k][0][sl][0] = inp[off];
        if (kBwd) reg[k][kArr - 1][sl][0] = dout[off];
      }
    }
    if constexpr (kBwd) {
      if constexpr (kVec) {
        const float4 w = *reinterpret_cast<const float4 *>(weight + col);
        wreg[k][0] = w.x, wreg[k][1] = w.y, wreg[k][2] = w.z, wreg[k][3] = w.w;
      } else {
        wreg[k][0] = weight[col];
      }
    }
  };
  auto store_tile = [&](int u, int k) {
    float *const T = tile + (u & 1) * kArr * kTileF;
#pragma unroll
    for (int sl = 0; sl < kSlots; sl++) {
      const int ri = slot_row(sl);
      if (ri < kExRows) {
        float t0[kW], t1[kW];
        if (kBwd) {
          const float2 st = stat[ri];
#pragma unroll
          for (int j = 0; j < kW; j++) {
            const float xh = (reg[k][0][sl][j] - st.x) * st.y;
            t0[j] = reg[k][kArr - 1][sl][j] * wreg[k][j];
            t1[j] = t0[j] * xh;
          }
        } else if (u < nt) {
#pragma unroll
          for (int j = 0; j < kW; j++) t0[j] = reg[k][0][sl][j];
        } else {
          const float m = stat[ri].x;
#pragma unroll
          for (int j = 0; j < kW; j++) {
            const float d = reg[k][0][sl][j] - m;
            t0[j] = d * d;
          }
        }
        float *const p = T + ri * kExPitch + lcol;
        if constexpr (kVec) {
          *reinterpret_cast<float4 *>(p) = make_float4(t0[0], t0[1], t0[2], t0[3]);
          if (kBwd) *reinterpret_cast<float4 *>(p + kTileF) = make_float4(t1[0], t1[1], t1[2], t1[3]);
        } else {
          p[0] = t0[0];
          if (kBwd) p[kTileF] = t1[0];
        }
      }
    }
  };
  if (wave > 0) {
#pragma unroll
    for (int k = 0; k < kExDepth; k++)
      if (k < nu) load_tile(k, k);
  }
  for (int u0 = 0; u0 < nu; u0 += kExDepth) {
#pragma unroll
    for (int k = 0; k < kExDepth; k++) {
      const int u = u0 + k;
      if (u >= nu) break;  // the same in every thread
      if (!kBwd && u == nt) {
        // the second pass's terms need the means: wavefront 0 has written them
        // after its last first-pass tile
        __syncthreads();
      }
      if (wave > 0) {
        store_tile(u, k);
        if (u + kExDepth < nu) load_tile(u + kExDepth, k);
      }
      // tile u is staged in buffer u & 1; the buffer written next round was
      // last read before this barrier
      __syncthreads();
      if (wave == 0) {
        const int cmax = min(kExTile, C - (u % nt) * kExTile);
        const float *X = tile + (u & 1) * kArr * kTileF + lane * kExPitch;
        if (cmax == kExTile) {
          const float4 *t[kArr];
#pragma unroll
          for (int a = 0; a < kArr; a++) t[a] = reinterpret_cast<const float4 *>(X + a * kTileF);
          chain_add4<kArr, kExBatch / kArr>(s, t, kExTile / 4);
        } else {
          for (int c = 0; c < cmax; c++) {
#pragma unroll
            for (int a = 0; a < kArr; a++) s[a] = s[a] + X[a * kTileF + c];
          }
        }
        if (!kBwd && u == nt - 1) {
          stat[lane].x = s[0] / Cf;
          s[0] = 0.0f;
        }
      }
    }
  }
  if (wave == 0) {
    if (kBwd) {
      rsum[lane] = make_float2(s[0] / Cf, s[kArr - 1] / Cf);
    } else {
      const float m = stat[lane].x;
      const float r = 1.0f / sqrtf(s[0] / Cf + 1e-5f);
      if (lane < kExRows && r0 + lane < rows) {
        mean[r0 + lane] = m;
        rstd[r0 + lane] = r;
      }
      stat[lane].y = r;
    }
  }
  __syncthreads();
  // the rows' elements, every wavefront on whole rows (inp and dout again,
  // from the cache), all the loads of a batch issued together
  for (int ri = wave; ri < kExRows; ri += kExLoaders + 1) {
    const int row = r0 + ri;
    if (row >= rows) break;
    const float m = stat[ri].x, r = stat[ri].y;
    const float2 rs = kBwd ? rsum[ri] : make_float2(0.0f, 0.0f);
    const size_t base = (size_t)row * C;
    if constexpr (kVec) {
      const int C4 = C >> 2;
      const float4 *x4 = reinterpret_cast<const float4 *>(inp + base);
      const float4 *y4 = reinterpret_cast<const float4 *>(kBwd ? dout + base : bias);
      const float4 *w4 = reinterpret_cast<const float4 *>(weight);
      float4 *o4 = reinterpret_cast<float4 *>(outp + base);
      for (int q0 = 0; q0 < C4; q0 += kExApplyVec * kWave) {
        float4 xv[kExApplyVec], wv[kExApplyVec], yv[kExApplyVec], dv[kExApplyVec];
#pragma unroll
        for (int k = 0; k < kExApplyVec; k++) {
          const int q = min(q0 + k * kWave + lane, C4 - 1);
          xv[k] = x4[q];
          wv[k] = w4[q];
          yv[k] = y4[q];
          if (kBwd) dv[k] = o4[q];
        }
#pragma unroll
        for (int k = 0; k < kExApplyVec; k++) {
          const int q = q0 + k * kWave + lane;
          if (q < C4) {
            float o[4];
#pragma unroll
            for (int j = 0; j < 4; j++) {
              const float xj = f4_get(xv[k], j), wj = f4_get(wv[k], j), yj = f4_get(yv[k], j);
              if (kBwd) {
                const float xh = (xj - m) * r;
                const float dn = yj * wj;
                o[j] = f4_get(dv[k], j) + r * (dn - rs.x - xh * rs.y);
              } else {
                o[j] = (xj - m) * r * wj + yj;
              }
            }
            o4[q] = make_float4(o[0], o[1], o[2], o[3]);
          }
        }
      }
    } else {
      for (int c0 = 0; c0 < C; c0 += kExApply * kWave) {
        float xv[kExApply], wv[kExApply], yv[kExApply], dv[kExApply];
#pragma unroll
        for (int k = 0; k < kExApply; k++) {
          const int c = min(c0 + k * kWave + lane, C - 1);
          xv[k] = inp[base + c];
          wv[k] = weight[c];
          yv[k] = kBwd ? dout[base + c] : bias[c];
          dv[k] = kBwd ? outp[base + c] : 0.0f;
        }
#pragma unroll
        for (int k = 0; k < kExApply; k++) {
          const int c = c0 + k * kWave + lane;
          if (c < C) {
            if (kBwd) {
              const float xh = (xv[k] - m) * r;
              const float dn = yv[k] * wv[k];
              outp[base + c] = dv[k] + r * (dn - rs.x - xh * rs.y);
            } else {
              outp[base + c] = (xv[k] - m) * r * wv[k] + yv[k];
            }
          }
        }
      }
    }
  }
}

template <bool kVec>
__device__ __forceinline__ void ln_cols_exact(float *lds, int blk, float *__restrict__ dweight,
                                              float *__restrict__ dbias, const float *__restrict__ dout,
                                              const float *__restrict__ inp, const float *__restrict__ mean,
                                              const float *__restrict__ rstd, int rows, int C) {
  constexpr int kTileF = kExChains * kExColPitch;
  constexpr int kSlots = kVec ? 1 : kExColSlots;
  constexpr int kW = kVec ? 4 : 1;  // floats per lane and slot
  float *const tile = lds;  // [2][kExChains][kExColPitch]: chain j's terms of the tile's rows
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & (kWave - 1);
  const int c0 = blk * kExCols;
  const int nt = (rows + kExColRows - 1) / kExColRows;
  // Loader lane L = 64 lw + lane. Scalar: slot sl holds tile row
  // 4 lw + 60 sl + lane / 16, column lane % 16. float4: tile row L / 4,
  // columns 4 (L % 4) + 0..3.
  const int lw = wave - 1;
  const int L = lw * kWave + lane;
  const int lc = kVec ? 4 * (L & 3) : (lane & (kExCols - 1));
  const int lcol = min(c0 + lc, C - kW);
  float rx[kExDepth][kSlots][kW], ry[kExDepth][kSlots][kW], rm[kExDepth][kSlots], rr[kExDepth][kSlots];
  auto tile_row = [&](int sl) {
    return kVec ? L >> 2 : (kWave / kExCols) * (lw + kExLoaders * sl) + lane / kExCols;
  };
  auto load_tile = [&](int t, int k) {
#pragma unroll
    for (int sl = 0; sl < kSlots; sl++) {
      const int row = min(t * kExColRows + tile_row(sl), rows - 1);
      const size_t off = (size_t)row * C + lcol;
      if constexpr (kVec) {
        const float4 x = *reinterpret_cast<const float4 *>(inp + off);
        const float4 y = *reinterpret_cast<const float4 *>(dout + off);
        rx[k][sl][0] = x.x, rx[k][sl][1] = x.y, rx[k][sl][2] = x.z, rx[k][sl][3] = x.w;
        ry[k][sl][0] = y.x, ry[k][sl][1] = y.y, ry[k][sl][2] = y.z, ry[k][sl][3] = y.w;
      } else {
        rx[k][sl][0] = inp[off];
        ry[k][sl][0] = dout[off];
      }
      rm[k][sl] = mean[row];
      rr[k][sl] = rstd[row];
    }
  };
  auto store_tile = [&](int t, int k) {
    float *const T = tile + (t & 1) * kTileF;
#pragma unroll
    for (int sl = 0; sl < kSlots; sl++) {
      const int ri = tile_row(sl);
#pragma unroll
      for (int j = 0; j < kW; j++) {
        const float xh = (rx[k][sl][j] - rm[k][sl]) * rr[k][sl];
        T[(lc + j) * kExColPitch + ri] = ry[k][sl][j] * xh;
        T[(kExCols + lc + j) * kExColPitch + ri] = ry[k][sl][j];
      }
    }
  };
  // the chain of wavefront 0's lane: dweight (lanes 0-15) or dbias (16-31) of
  // column c0 + lane % 16; lanes 32-63 follow a copy and store nothing
  const bool chain = wave == 0 && lane < kExChains;
  const int cc = c0 + (lane & (kExCols - 1));
  float *const dst = (lane < kExCols ? dweight : dbias) + min(cc, C - 1);
  float acc[1] = {chain ? *dst : 0.0f};
  if (wave > 0) {
#pragma unroll
    for (int k = 0; k < kExDepth; k++)
      if (k < nt) load_tile(k, k);
  }
  for (int t0 = 0; t0 < nt; t0 += kExDepth) {
#pragma unroll
    for (int k = 0; k < kExDepth; k++) {
      const int t = t0 + k;
      if (t >= nt) break;  // the same in every thread
      if (wave > 0) {
        store_tile(t, k);
        if (t + kExDepth < nt) load_tile(t + kExDepth, k);
      }
      __syncthreads();
      if (wave == 0) {
        const float *T = tile + (t & 1) * kTileF + (lane & (kExChains - 1)) * kExColPitch;
        const int rmax = min(kExColRows, rows - t * kExColRows);
        if (rmax == kExColRows) {
          const float4 *t4[1] = {reinterpret_cast<const float4 *>(T)};
          chain_add4<1, kExColBatch>(acc, t4, kExColRows / 4);
        } else {
          for (int i = 0; i < rmax; i++) acc[0] = acc[0] + T[i];
        }
      }
    }
  }
  if (chain && cc < C) *dst = acc[0];
}

template <bool kVec>
__global__ __launch_bounds__(kExThreads) void k_ln_fwd_exact(float *__restrict__ out, float *__restrict__ mean,
                                                             float *__restrict__ rstd, const float *__restrict__ inp,
                                                             const float *__restrict__ weight,
                                                             const float *__restrict__ bias, int rows, int C) {
  __shared__ __align__(16) float lds[ex_row_lds(1)];
  ln_rows_exact<false, kVec>(lds, blockIdx.x, out, mean, rstd, inp, nullptr, weight, bias, rows, C);
}

// workgroups [0, nrow) the rows (dinp), the others the columns (dweight, dbias)
template <bool kVec>
__global__ __launch_bounds__(kExThreads) void k_ln_bwd_exact(float *__restrict__ dinp, float *__restrict__ dweight,
                                                             float *__restrict__ dbias, const float *__restrict__ dout,
                                                             const float *__restrict__ inp,
                                                             const float *__restrict__ weight,
                                                             const float *__restrict__ mean,
                                                             const float *__restrict__ rstd, int rows, int C,
                                                             int nrow) {
  __shared__ __align__(16) float lds[kExBwdLds];
  if ((int)blockIdx.x < nrow)
    ln_rows_exact<true, kVec>(lds, blockIdx.x, dinp, const_cast<float *>(mean), const_cast<float *>(rstd), inp, dout,
                              weight, nullptr, rows, C);
  else
    ln_cols_exact<kVec>(lds, (int)blockIdx.x - nrow, dweight, dbias, dout, inp, mean, rstd, rows, C);
}

}  // namespace

namespace {
std::atomic<int> g_ln_exact{0};
}  // namespace

void set_layernorm_exact(int on) { g_ln_exact.store(on ? 1 : 0); }
int layernorm_exact() { return g_ln_exact.load(); }

int launch_layernorm_forward_exact(float *out, float *mean, float *rstd, const float *inp, const float *weight,
                                   const float *bias, int rows, int C) {
  if (rows == 0 || C == 0) return 0;
  const bool vec = C % 4 == 0 && aligned16(out) && aligned16(inp) && aligned16(weight) && aligned16(bias);
  const dim3 grid(grid_for((size_t)rows, kExRows)), block(kExThreads);
  if (vec)
    launch(k_ln_fwd_exact<true>, grid, block, 0, out, mean, rstd, inp, weight, bias, rows, C);
  else
    launch(k_ln_fwd_exact<false>, grid, block, 0, out, mean, rstd, inp, weight, bias, rows, C);
  return check_launch("layernorm_forward (exact)");
}

namespace {
// Whether a backward writes over its own dout or inp (dinp = dout, say). A
// row's terms are then those of the arrays as they were, so the kernels whose
// column workgroups run beside the row workgroups (few rows, and the exact
// form) cannot take the call as it is, and the lane loops sum the columns first.
// The others read all of a row, and add its column terms in registers, before
// they write it.
bool in_place(const float *dinp, const float *dx, const float *dy, const float *dout, const float *inp, size_t n) {
  const auto overlap = [n](const float *a, const float *b) {
    const uintptr_t x = (uintptr_t)a, y = (uintptr_t)b;
    return a && (x < y ? y - x : x - y) < n * sizeof(float);
  };
  for (const float *w : {dinp, dx, dy})
    if (overlap(w, dout) || overlap(w, inp)) return true;
  return false;
}
}  // namespace

int launch_layernorm_backward_exact(float *dinp, float *dweight, float *dbias, const float *dout, const float *inp,
                                    const float *weight, const float *mean, const float *rstd, int rows, int C) {
  if (rows == 0 || C == 0) return 0;
  const bool vec = C % 4 == 0 && aligned16(dinp) && aligned16(dout) && aligned16(inp) && aligned16(weight);
  const int nrow = (int)grid_for((size_t)rows, kExRows), ncol = (int)grid_for((size_t)C, kExCols);
  const auto go = [&](int blocks, int row_blocks) {
    launch(vec ? k_ln_bwd_exact<true> : k_ln_bwd_exact<false>, dim3(blocks), dim3(kExThreads), 0, dinp, dweight, dbias,
           dout, inp, weight, mean, rstd, rows, C, row_blocks);
  };
  if (in_place(dinp, nullptr, nullptr, dout, inp, (size_t)rows * C)) {
    go(ncol, 0);  // all columns before any row is written
    go(nrow, nrow);
  } else {
    go(nrow + ncol, nrow);
  }
  return check_launch("layernorm_backward (exact)");
}

int launch_layernorm_forward(float *out, float *mean, float *rstd, const float *inp,
                             const float *weight, const float *bias, int rows, int C) {
  if (rows == 0) return 0;
  if (layernorm_exact()) return launch_layernorm_forward_exact(out, mean, rstd, inp, weight, bias, rows, C);
  if (row_in_wave(C) || row_in_block(C)) {
    launch_ln_fwd_rows<false>(out, mean, rstd, inp, weight, bias, rows, C, nullptr, nullptr);
  } else {
    const dim3 grid(grid_for((size_t)rows, kWavesPerBlock)), block(kBlock);
    launch(k_ln_fwd_scalar, grid, block, 0, out, mean, rstd, inp, weight, bias,
                       rows, C);
  }
  return check_launch("layernorm_forward");
}

namespace {
// tail: the workgroups finish the column sums into dweight/dbias themselves
// (ln_bwd_tail); only for the per-op modes (dinp read and written, residual
// targets read).
template <bool kRes, int kDinp, bool kAssign>
int launch_ln_bwd_vec(float *dinp, float *partial, const float *dout, const float *inp,
                      const float *weight, const float *mean, const float *rstd, int rows, int C,
                      float *rdx, float *rdy, int max_blocks, bool tail = false, float *dweight = nullptr,
                      float *dbias = nullptr) {
  static_assert(kRes || (kDinp == kDinpRw && !kAssign), "the plain backward reads and writes dinp");
  constexpr bool kTailOk = kDinp == kDinpRw && !kAssign;
  int nblk, rpw;
  const int V = slots_of(C, kWave);
  const int same = rdx == rdy ? 1 : 0;
  const bool nt = (size_t)rows * (size_t)C < ((size_t)1 << 21);
  // the kernel with and without the in-launch column sums
  const auto both = [&](auto k_plain, auto k_tail, dim3 grid, dim3 block, int rp) {
    if (kTailOk && tail)
      launch(k_tail, grid, block, 0, dinp, partial, dout, inp, weight, mean, rstd, rows, C, rp, rdx, rdy, same,
             dweight, dbias);
    else
      launch(k_plain, grid, block, 0, dinp, partial, dout, inp, weight, mean, rstd, rows, C, rp, rdx, rdy, same,
             nullptr, nullptr);
  };
  if (team_path(rows, C)) {
    int rpt;
    team_shape(rows, max_blocks, &nblk, &rpt);
    const dim3 grid(nblk), block(kTeamParts * kTeams * kWave);
    if constexpr (kRes)
      both(k_ln_bwd_team<kTeamParts, kTeams, 4, true, 3, true, kDinp, kAssign, false>,
           k_ln_bwd_team<kTeamParts, kTeams, 4, true, 3, true, kDinp, kAssign, kTailOk>, grid, block, rpt);
    else if (nt)
      both(k_ln_bwd_team<kTeamParts, kTeams, 2, false, 1, true, kDinpRw, false, false>,
           k_ln_bwd_team<kTeamParts, kTeams, 2, false, 1, true, kDinpRw, false, true>, grid, block, rpt);
    else
      both(k_ln_bwd_team<kTeamParts, kTeams, 2, false, 1, false, kDinpRw, false, false>,
           k_ln_bwd_team<kTeamParts, kTeams, 2, false, 1, false, kDinpRw, false, true>, grid, block, rpt);
    return nblk;
  }
  const BwdCfg k = bwd_cfg(V, kRes);
  bwd_shape_vec(rows, k, max_blocks, &nblk, &rpw);
  const dim3 grid(nblk), block(k.W * kWave);
  const bool rag = (C & 3) != 0;  // takes only the modes of the per-op calls (kTailOk)
  switch (V) {
#define UGK_LN_BWD_K(v, ntv, tl)                                                                                    \
  k_ln_bwd_vec<v, bwd_cfg(v, kRes).W, bwd_cfg(v, kRes).R, kRes, bwd_cfg(v, kRes).MINW, ntv, kDinp, kAssign, tl, false>
#define UGK_LN_BWD(v)                                                                                               \
  case v:                                                                                                           \
    if (rag) {                                                                                                      \
      if constexpr (kTailOk)                                                                                        \
        launch(k_ln_bwd_vec<v, bwd_cfg(v, kRes).W, bwd_cfg(v, kRes).R, kRes, bwd_cfg(v, kRes).MINW, true, kDinpRw,   \
                            false, false, true>,                                                                    \
               grid, block, 0, dinp, partial, dout, inp, weight, mean, rstd, rows, C, rpw, rdx, rdy, same, nullptr, \
               nullptr);                                                                                            \
    } else if (kRes || nt)                                                                                          \
      both(UGK_LN_BWD_K(v, true, false), UGK_LN_BWD_K(v, true, kTailOk), grid, block, rpw);                         \
    else                                                                                                            \
      both(UGK_LN_BWD_K(v, kRes, false), UGK_LN_BWD_K(v, kRes, kTailOk), grid, block, rpw);                         \
    break;
    UGK_LN_BWD(1) UGK_LN_BWD(2) UGK_LN_BWD(3) UGK_LN_BWD(4)
    UGK_LN_BWD(5) UGK_LN_BWD(6) UGK_LN_BWD(7) UGK_LN_BWD(8)
#undef UGK_LN_BWD
#undef UGK_LN_BWD_K
  }
  return nblk;
}

// Whether the per-op backward finishes its column sums in the main launch (1)
// or in a second one (0, the default: faster, see ln_bwd_tail); both give the
// same bits.
std::atomic<int> g_ln_tail{0};
}  // namespace

void set_layernorm_tail(int on) { g_ln_tail.store(on ? 1 : 0); }
int layernorm_tail() { return g_ln_tail.load(); }

namespace {
// The backward of small_path: the column totals are added to dweight
// and dbias, or stored there (add false), or left out (dweight null).
template <bool kRes>
void launch_ln_bwd_small(float *dinp, float *dweight, float *dbias, bool add, float *dx, float *dy, const float *dout,
                         const float *inp, const float *weight, const float *mean, const float *rstd, int rows, int C,
                         LnBwdMode md) {
  const bool wide = row_in_block(C);
  const int ncol = dweight ? (int)grid_for((size_t)C, kSmallCols) : 0;
  const int nrow = wide ? rows : (int)grid_for((size_t)rows, kWavesPerBlock);
  const auto go = [&](auto k) {
    launch(k, dim3(ncol + nrow), dim3(kBlock), 0, dinp, dweight, dbias, dout, inp, weight, mean, rstd, rows, C, ncol,
           add ? 1 : 0, dx, dy, md);
  };
  switch (slots_of(C, wide ? kBlock : kWave)) {
#define UGK_LN_SMALL(v)                              \
  case v:                                            \
    if (wide) go(k_ln_bwd_small<v, kWavesPerBlock, kRes>); \
    else go(k_ln_bwd_small<v, 1, kRes>);             \
    break;
    UGK_LN_SMALL(1) UGK_LN_SMALL(2) UGK_LN_SMALL(3) UGK_LN_SMALL(4)
    UGK_LN_SMALL(5) UGK_LN_SMALL(6) UGK_LN_SMALL(7) UGK_LN_SMALL(8)
#undef UGK_LN_SMALL
  }
}

template <bool kRes>
void launch_ln_bwd_wide(float *dinp, float *partial, float *dx, float *dy, const float *dout, const float *inp,
                        const float *weight, const float *mean, const float *rstd, int rows, int C, int max_blocks,
                        LnBwdMode md, int *nblk) {
  int rpw;
  wide_shape(rows, max_blocks, nblk, &rpw);
  const auto go = [&](auto k) {
    launch(k, dim3(*nblk), dim3(kWideWaves * kWave), 0, dinp, partial, dout, inp, weight, mean, rstd, rows, C, rpw, dx,
           dy, md);
  };
  const int V = slots_of(C, kWideWaves * kWave);
  if (V <= 2) go(k_ln_bwd_wide<2, kWideWaves, 2, kRes>);
  else if (V == 3) go(k_ln_bwd_wide<3, kWideWaves, 1, kRes>);
  else go(k_ln_bwd_wide<4, kWideWaves, 1, kRes>);
}
}  // namespace

int launch_layernorm_backward_partials(float *dinp, float *partial, LnCols cols, float *dweight, float *dbias,
                                       float *dx, float *dy, const float *dout, const float *inp,
                                       const float *weight, const float *mean, const float *rstd, int rows, int C,
                                       int max_blocks, int *nblk, int dinp_mode, bool assign_res) {
  *nblk = 0;
  if (rows == 0) return 0;
  const bool res = dx != nullptr;
  if (!(res && dinp_mode == kDinpNone ? assign_res : !assign_res || (res && dinp_mode == kDinpRead)))
    return set_error(UGK_EINVAL, "layernorm_backward: unsupported dinp mode %d with assign %d", dinp_mode,
                     (int)assign_res);
  const LnBwdMode md{dinp_mode != kDinpNone, dinp_mode == kDinpRw, assign_res, dx == dy};
  if (small_path(rows, C, dout, inp) && !in_place(dinp, dx, dy, dout, inp, (size_t)rows * C)) {
    const bool add = cols == kColsAdd;
    float *const g = add ? dweight : cols == kColsPartial ? partial : nullptr, *const b = add ? dbias : partial + C;
    if (res)
      launch_ln_bwd_small<true>(dinp, g, b, add, dx, dy, dout, inp, weight, mean, rstd, rows, C, md);
    else
      launch_ln_bwd_small<false>(dinp, g, b, add, dx, dy, dout, inp, weight, mean, rstd, rows, C, md);
    if (cols == kColsPartial) *nblk = 1;
    return check_launch("layernorm_backward");
  }
  if (row_in_wave(C)) {
    // ragged rows have the kernels of the per-op modes only, which read and write everything
    const int mode = (C & 3) != 0 ? kDinpRw : dinp_mode;
    const bool assign = (C & 3) == 0 && assign_res;
#define UGK_LN_BWD_MODE(d, a) \
  launch_ln_bwd_vec<true, d, a>(dinp, partial, dout, inp, weight, mean, rstd, rows, C, dx, dy, max_blocks)
    if (!res)
      *nblk = launch_ln_bwd_vec<false, kDinpRw, false>(dinp, partial, dout, inp, weight, mean, rstd, rows, C,
                                                       nullptr, nullptr, max_blocks);
    else if (mode == kDinpRw)
      *nblk = UGK_LN_BWD_MODE(kDinpRw, false);
    else if (mode == kDinpNone)
      *nblk = UGK_LN_BWD_MODE(kDinpNone, true);
    else if (assign)
      *nblk = UGK_LN_BWD_MODE(kDinpRead, true);
    else
      *nblk = UGK_LN_BWD_MODE(kDinpRead, false);
#undef UGK_LN_BWD_MODE
    return check_launch("layernorm_backward");
  }
  if (row_in_block(C)) {
    if (res)
      launch_ln_bwd_wide<true>(dinp, partial, dx, dy, dout, inp, weight, mean, rstd, rows, C, max_blocks, md, nblk);
    else
      launch_ln_bwd_wide<false>(dinp, partial, dx, dy, dout, inp, weight, mean, rstd, rows, C, max_blocks, md, nblk);
    return check_launch("layernorm_backward");
  }
  int rpb;
  bwd_shape(rows, max_blocks < kMaxScalarBlocks ? max_blocks : kMaxScalarBlocks, nblk, &rpb);
  launch(in_place(dinp, nullptr, nullptr, dout, inp, (size_t)rows * C) ? k_ln_bwd_scalar<true> : k_ln_bwd_scalar<false>,
         dim3(*nblk), dim3(kBlock), 0, dinp, partial, dout, inp, weight, mean, rstd, rows, C, rpb);
  if (int e = check_launch("layernorm_backward")) return e;
  return res ? launch_residual_backward(dx, dy, dinp, (size_t)rows * C) : 0;
}

int launch_layernorm_reduce(const LnReduceJob *jobs, int njobs, int rows, int C) {
  LnReduceBatch sums{}, cols{};  // jobs with partial rows, and without
  int nsums = 0, ncols = 0;
  for (int j = 0; j < njobs; j++) {
    const bool later = jobs[j].nblk == 0, last = j + 1 == njobs;
    if (later) cols.job[ncols++] = jobs[j];
    else sums.job[nsums++] = jobs[j];
    if (nsums == kMaxReduceJobs || (last && nsums > 0)) {
      launch(k_ln_bwd_reduce_batch, dim3(grid_for((size_t)2 * C, kRedCols), nsums), dim3(kRedCols * kRedGroups), 0,
             sums, C);
      nsums = 0;
    }
    if (ncols == kMaxReduceJobs || (last && ncols > 0)) {
      launch(k_ln_small_cols_batch, dim3(grid_for((size_t)C, kSmallCols), ncols), dim3(kBlock), 0, cols, rows, C);
      ncols = 0;
    }
  }
  return check_launch("layernorm_backward (column sums)");
}

int launch_layernorm_residual_backward_into(float *partial, int max_blocks, float *dinp, float *dweight,
                                            float *dbias, float *dx, float *dy, const float *dout,
                                            const float *inp, const float *weight, const float *mean,
                                            const float *rstd, int rows, int C) {
  if (rows == 0) return 0;
  const bool res = dx != nullptr;
  if (layernorm_exact()) {  // no partial rows: the exact kernels keep their chains in LDS and registers
    if (int e = launch_layernorm_backward_exact(dinp, dweight, dbias, dout, inp, weight, mean, rstd, rows, C))
      return e;
    return res ? launch_residual_backward(dx, dy, dinp, (size_t)rows * C) : 0;
  }
  if (layernorm_tail() && row_in_wave(C) && (C & 3) == 0 && !small_path(rows, C, dout, inp)) {
    if (res)
      launch_ln_bwd_vec<true, kDinpRw, false>(dinp, partial, dout, inp, weight, mean, rstd, rows, C, dx, dy,
                                              max_blocks, true, dweight, dbias);
    else
      launch_ln_bwd_vec<false, kDinpRw, false>(dinp, partial, dout, inp, weight, mean, rstd, rows, C, nullptr,
                                               nullptr, max_blocks, true, dweight, dbias);
    return check_launch("layernorm_backward");
  }
  int nblk;
  if (int e = launch_layernorm_backward_partials(dinp, partial, kColsAdd, dweight, dbias, dx, dy, dout, inp, weight,
                                                 mean, rstd, rows, C, max_blocks, &nblk))
    return e;
  if (nblk == 0) return 0;  // the launch has added the column sums
  const LnReduceJob job{partial, dweight, dbias, nblk, dout, inp, mean, rstd};
  return launch_layernorm_reduce(&job, 1, rows, C);
}

int launch_layernorm_residual_backward(float *dinp, float *dweight, float *dbias, float *dx, float *dy,
                                       const float *dout, const float *inp, const float *weight,
                                       const float *mean, const float *rstd, int rows, int C) {
  if (rows == 0) return 0;
  float *partial = static_cast<float *>(workspace(kRegLn, layernorm_backward_scratch(rows, C)));
  if (!partial) return UGK_ENOMEM;
  // the workspace holds the bound's number of partial rows, and no shape takes
  // more workgroups than the cap it is given
  return launch_layernorm_residual_backward_into(partial, layernorm_backward_blocks_bound(rows, C), dinp, dweight,
                                                 dbias, dx, dy, dout, inp, weight, mean, rstd, rows, C);
}

// ---- allocation-free variant ------------------------------------------------
// The partial rows in a file-scope device array (one copy per GPU, held until
// the process ends) instead of the workspace. Host code never passes the
// array's name to a kernel (on the host it stands for a host-side shadow):
// it looks up the array's device address once per device with
// hipGetSymbolAddress and passes that.
}  // namespace ugk

static __device__ __align__(256) float scratch[ugk::kNoAllocScratchBytes / sizeof(float)];

namespace ugk {
namespace {
struct NoAllocAddr {
  float *ptr = nullptr;
  hipError_t err = hipSuccess;
  bool looked_up = false;
};
NoAllocAddr g_noalloc[64];
std::mutex g_noalloc_mu;
}  // namespace

float *noalloc_scratch() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) {
    (void)hipGetLastError();
    set_error(UGK_EHIP, "no-alloc scratch: hipGetDevice failed");
    return nullptr;
  }
  std::lock_guard<std::mutex> lock(g_noalloc_mu);
  NoAllocAddr &a = g_noalloc[dev];
  if (!a.looked_up) {  // once per device, with that device current
    void *p = nullptr;
    a.err = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (a.err != hipSuccess) (void)hipGetLastError();
    a.ptr = a.err == hipSuccess ? static_cast<float *>(p) : nullptr;
    a.looked_up = true;
  }
  if (!a.ptr) set_error(UGK_EHIP, "no-alloc scratch: hipGetSymbolAddress failed: %s", hipGetErrorString(a.err));
  return a.ptr;
}

int noalloc_max_blocks(int C) {
  const size_t per_row = 2 * (size_t)C * sizeof(float);
  const size_t fit = kNoAllocScratchBytes / per_row;
  return fit < (size_t)kMaxPartialRows ? (int)fit : kMaxPartialRows;
}

int launch_layernorm_backward(float *dinp, float *dweight, float *dbias, const float *dout,
                              const float *inp, const float *weight, const float *mean,
                              const float *rstd, int rows, int C) {
  return launch_layernorm_residual_backward(dinp, dweight, dbias, nullptr, nullptr, dout, inp, weight, mean,
                                            rstd, rows, C);
}

}  // namespace ugk
