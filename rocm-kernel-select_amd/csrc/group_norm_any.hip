// GroupNorm forward where the aligned kernels of group_norm.hip do not apply: NC[S] rows that are
// no multiple of 16 bytes (odd image sizes, misaligned views), and channels-last tensors whose
// groups or channel counts do not fit its column map.  HBM-bound like those.
#include <algorithm>

#include "gn_any.h"
#include "param_loads.h"

namespace atk {

namespace {

// 16 bytes at an element-aligned address: one instruction each (unaligned global access).
typedef unsigned int u32x4_u __attribute__((ext_vector_type(4), aligned(2)));
__device__ __forceinline__ uint4 ld16u(const void* p) {
  const u32x4_u v = *reinterpret_cast<const u32x4_u*>(p);
  return make_uint4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ void st16u_nt(void* p, uint4 r) {
  const u32x4_u v = {r.x, r.y, r.z, r.w};
  __builtin_nontemporal_store(v, reinterpret_cast<u32x4_u*>(p));
}

// ---------------------------------------------------------------------------------------
// NC[S] rows of any length.  A group is E = cpg * S consecutive elements, read as 16-byte vectors
// from its first element on, whatever its address; the last vector, where E is no multiple of
// one, is read as the group's last 16 bytes.  Elements that it shares with the vector before are
// left out of the sums, and stored twice with the same value where the group is held in
// registers, once where it is read again.  y may be x.
// ---------------------------------------------------------------------------------------
constexpr int GA_AFF = 1024;  // channels per group whose scale and shift fit LDS
constexpr int GA_NT = 256;    // threads of the two-pass kernels

struct GaArgs {
  const void* x;
  const void* gamma;
  const void* beta;
  void* y;
  int64_t E;
  uint32_t S, cpg, G;
  float eps;
  int pdt;
  FastDiv div_s;
  float* partials;  // [ngroups][NS] (mean, M2)
  int NS;
  int64_t slice;
};

__device__ __forceinline__ void affine_of(const GaArgs& a, int64_t c, float mean, float rstd, float& sc, float& sh) {
  const float gm = a.gamma ? load_param(a.gamma, a.pdt, c) : 1.f;
  const float bt = a.beta ? load_param(a.beta, a.pdt, c) : 0.f;
  sc = rstd * gm;
  sh = bt - mean * sc;
}

// Running sums of one vector about the shift K; elements below `skip` are left out.
template <typename T, bool MASK>
__device__ __forceinline__ void add_vec(const Vec16<T>& v, float K, int skip, float& s1, float& s2) {
#pragma unroll
  for (int k = 0; k < Vec16<T>::N; ++k) {
    float d = to_f32(v.e[k]) - K;
    if (MASK) d = k >= skip ? d : 0.f;
    s1 += d;
    s2 = fmaf(d, d, s2);
  }
}

// n, K, s1, s2 of every thread -> mean and M2 over the block (exact merge of the threads' means).
template <int NT>
__device__ __forceinline__ void merge_block(float n, float K, float s1, float s2, float total, float* red, float& mean,
                                            float& m2) {
  float mt = 0.f, qt = 0.f;
  if (n > 0.f) {
    const float q = s1 / n;
    mt = K + q;
    qt = fmaxf(fmaf(-s1, q, s2), 0.f);
  }
  mean = block_sum<NT>(n * mt, red) / total;
  const float d = mt - mean;
  m2 = block_sum<NT>(fmaf(n * d, d, qt), red);
}

// y of one vector whose first element is group element e: at most one channel boundary lies
// inside it (S >= VEC).  aff(c): scale and shift of the group's channel c.
template <typename T, bool SILU, typename Aff>
__device__ __forceinline__ uint4 apply_vec(const Vec16<T>& v, uint32_t e, const GaArgs& a, Aff aff) {
  constexpr int VEC = Vec16<T>::N;
  const uint32_t c = fdiv(e, a.div_s);
  const int b = (int)((c + 1) * a.S - e);  // elements before the next channel
  float sc, sh, o[VEC];
  aff(c, sc, sh);
#pragma unroll
  for (int k = 0; k < VEC; ++k) o[k] = fmaf(to_f32(v.e[k]), sc, sh);
  if (b < VEC) {
    aff(c + 1, sc, sh);
#pragma unroll
    for (int k = 1; k < VEC; ++k) o[k] = k >= b ? fmaf(to_f32(v.e[k]), sc, sh) : o[k];
  }
  if constexpr (SILU) {
#pragma unroll
    for (int k = 0; k < VEC; ++k) o[k] = silu_f32(o[k]);
  }
  return pack16<T>(o);
}

// One workgroup per group, which it holds in registers: x is read once.
template <typename T, int NT, int EPV, bool SILU>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4))) void gn_any_resident_kernel(GaArgs a) {
  constexpr int VEC = Vec16<T>::N;
  __shared__ float red[NT / 64];
  __shared__ float aff[2 * GA_AFF];
  const int tid = threadIdx.x;
  const int64_t gi = blockIdx.x;
  const int E = (int)a.E;
  const T* __restrict__ xg = static_cast<const T*>(a.x) + gi * a.E;
  T* __restrict__ yg = static_cast<T*>(a.y) + gi * a.E;
  const int nvec = (E + VEC - 1) / VEC, last = (nvec - 1) / NT;  // vector row that holds the last vector
  Vec16<T> buf[EPV];
#pragma unroll
  for (int i = 0; i < EPV; ++i)
    if (i <= last) buf[i].raw = ld16u(xg + min((i * NT + tid) * VEC, E - VEC));
  const int64_t c0 = (int64_t)(gi % a.G) * a.cpg;
  const float K = to_f32(buf[0].e[0]);
  float s1 = 0.f, s2 = 0.f, n = 0.f;
#pragma unroll
  for (int i = 0; i < EPV; ++i) {
    // converted only after the vector before it is summed (left free, all of them are held in fp32)
    asm volatile("" : "+v"(buf[i].raw.x), "+v"(buf[i].raw.y), "+v"(buf[i].raw.z), "+v"(buf[i].raw.w), "+v"(s1), "+v"(s2));
    if (i < last) {
      add_vec<T, false>(buf[i], K, 0, s1, s2);
      n += VEC;
    } else if (i == last) {
      const int e = (i * NT + tid) * VEC, skip = min(max(e - (E - VEC), 0), VEC);
      add_vec<T, true>(buf[i], K, skip, s1, s2);
      n += VEC - skip;
    }
  }
  float mean, m2;
  merge_block<NT>(n, K, s1, s2, (float)E, red, mean, m2);
  const float rstd = 1.0f / sqrtf(m2 / (float)E + a.eps);
  for (int c = tid; c < (int)a.cpg; c += NT) affine_of(a, c0 + c, mean, rstd, aff[c], aff[GA_AFF + c]);
  __syncthreads();
#pragma unroll
  for (int i = 0; i < EPV; ++i) {
    if (i > last) break;
    asm volatile("" : "+v"(buf[i].raw.x), "+v"(buf[i].raw.y), "+v"(buf[i].raw.z), "+v"(buf[i].raw.w));
    if (i * NT + tid >= nvec) continue;
    const int e = min((i * NT + tid) * VEC, E - VEC);
    st16u_nt(yg + e, apply_vec<T, SILU>(buf[i], (uint32_t)e, a, [&](uint32_t c, float& sc, float& sh) {
               sc = aff[c];
               sh = aff[GA_AFF + c];
             }));
  }
}

// Larger groups: slice statistics, then a pass that merges them and normalises.
template <typename T>
__global__ __launch_bounds__(GA_NT) void gn_any_stats_kernel(GaArgs a) {
  constexpr int VEC = Vec16<T>::N, U = 4;
  __shared__ float red[GA_NT / 64];
  const int64_t gi = blockIdx.x / a.NS, s = blockIdx.x - gi * a.NS;
  const int64_t s0 = s * a.slice, s1_ = min(s0 + a.slice, a.E);
  const T* __restrict__ xg = static_cast<const T*>(a.x) + gi * a.E;
  float K = 0.f, s1 = 0.f, s2 = 0.f, n = 0.f;
  for (int64_t e0 = s0 + (int64_t)threadIdx.x * VEC; e0 < s1_; e0 += (int64_t)U * GA_NT * VEC) {
    Vec16<T> v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u].raw = ld16u(xg + min(e0 + (int64_t)u * GA_NT * VEC, a.E - VEC));
    if (n == 0.f) K = to_f32(v[0].e[VEC - 1]);  // in the slice also where the vector was moved down
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t e = e0 + (int64_t)u * GA_NT * VEC;
      const int skip = e >= s1_ ? VEC : (int)max(e - (a.E - VEC), (int64_t)0);
      add_vec<T, true>(v[u], K, skip, s1, s2);
      n += VEC - skip;
    }
  }
  float mean, m2;
  merge_block<GA_NT>(n, K, s1, s2, (float)(s1_ - s0), red, mean, m2);
  if (threadIdx.x == 0) {
    a.partials[(gi * a.NS + s) * 2] = mean;
    a.partials[(gi * a.NS + s) * 2 + 1] = m2;
  }
}

template <typename T, bool SILU>
__global__ __launch_bounds__(GA_NT) void gn_any_apply_kernel(GaArgs a) {
  constexpr int VEC = Vec16<T>::N, U = 4;
  __shared__ float st[2];
  const int tid = threadIdx.x;
  const int64_t gi = blockIdx.x / a.NS, s = blockIdx.x - gi * a.NS;
  const int64_t s0 = s * a.slice, s1 = min(s0 + a.slice, a.E);
  const T* xg = static_cast<const T*>(a.x) + gi * a.E;
  T* yg = static_cast<T*>(a.y) + gi * a.E;
  Vec16<T> v[U];
  auto issue = [&](int64_t e0) {
#pragma unroll
    for (int u = 0; u < U; ++u) v[u].raw = ld16u(xg + min(e0 + (int64_t)u * GA_NT * VEC, a.E - VEC));
  };
  const int64_t first = s0 + (int64_t)tid * VEC;
  issue(first);  // does not depend on the statistics
  if (tid < 64) {
    const float* p = a.partials + gi * (int64_t)a.NS * 2;
    auto len = [&](int i) { return (float)(min((int64_t)(i + 1) * a.slice, a.E) - (int64_t)i * a.slice); };
    float sm = 0.f, q = 0.f;
    for (int i = tid; i < a.NS; i += 64) sm += len(i) * p[2 * i];
    const float mean = wave_sum(sm) / (float)a.E;
    for (int i = tid; i < a.NS; i += 64) {
      const float d = p[2 * i] - mean;
      q += p[2 * i + 1] + len(i) * d * d;
    }
    q = wave_sum(q);
    if (tid == 0) {
      st[0] = mean;
      st[1] = 1.0f / sqrtf(q / (float)a.E + a.eps);
    }
  }
  __syncthreads();
  const float mean = st[0], rstd = st[1];
  const int64_t c0 = (int64_t)(gi % a.G) * a.cpg;
  for (int64_t e0 = first; e0 < s1; e0 += (int64_t)U * GA_NT * VEC) {
    if (e0 != first) issue(e0);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t e = e0 + (int64_t)u * GA_NT * VEC, em = min(e, a.E - VEC);
      if (e >= s1) continue;
      Vec16<T> o;
      o.raw = apply_vec<T, SILU>(v[u], (uint32_t)em, a, [&](uint32_t c, float& sc, float& sh) {
        affine_of(a, c0 + c, mean, rstd, sc, sh);
      });
      if (em == e) {
        st16u_nt(yg + e, o.raw);
      } else {  // the elements shared with the vector before belong to its thread: y may be x, normalised there already
        const int own = (int)(e - em);
#pragma unroll
        for (int k = 1; k < VEC; ++k)
          if (k >= own) yg[em + k] = o.e[k];
      }
    }
  }
}

template <typename T, int NT, int EPV>
int launch_resident(const GaArgs& a, int64_t ngroups, int silu, hipStream_t s) {
  if (silu) hipLaunchKernelGGL((gn_any_resident_kernel<T, NT, EPV, true>), dim3((unsigned)ngroups), dim3(NT), 0, s, a);
  else hipLaunchKernelGGL((gn_any_resident_kernel<T, NT, EPV, false>), dim3((unsigned)ngroups), dim3(NT), 0, s, a);
  return check_launch("gn_any_resident_kernel");
}

template <typename T>
int launch_any(const GaArgs& a, int64_t ngroups, int silu, hipStream_t s) {
  constexpr int VEC = 16 / sizeof(T);
  const int64_t nvec = (a.E + VEC - 1) / VEC;
  // Up to 8192 vectors a group stay in one workgroup's registers; larger ones take two passes.
  // With fewer groups than keep four small workgroups on every CU, a group gets as many threads
  // as leave two vectors each: one wave's loads in flight do not fill a CU ([8, 256, 45, 45]
  // bf16, 256 groups of 2025 vectors: 10.3 us with 256 threads, 7.7 us with 1024).
  if (a.cpg <= GA_AFF && nvec <= 8192 && ngroups <= 0x7fffffff) {
    if (nvec <= 512) return launch_resident<T, 256, 2>(a, ngroups, silu, s);
    if (ngroups >= 4 * device_cu_count()) {
      if (nvec <= 1024) return launch_resident<T, 256, 4>(a, ngroups, silu, s);
      if (nvec <= 2048) return launch_resident<T, 256, 8>(a, ngroups, silu, s);
      if (nvec <= 4096) return launch_resident<T, 512, 8>(a, ngroups, silu, s);
    }
    if (nvec <= 1024) return launch_resident<T, 512, 2>(a, ngroups, silu, s);
    if (nvec <= 2048) return launch_resident<T, 1024, 2>(a, ngroups, silu, s);
    if (nvec <= 4096) return launch_resident<T, 1024, 4>(a, ngroups, silu, s);
    return launch_resident<T, 1024, 8>(a, ngroups, silu, s);
  }
  const int64_t nblk = ngroups * a.NS;
  if (nblk > 0x7fffffff) return fail(ATK_UNSUPPORTED, "group_norm: grid too large");
  hipLaunchKernelGGL((gn_any_stats_kernel<T>), dim3((unsigned)nblk), dim3(GA_NT), 0, s, a);
  const int rc = check_launch("gn_any_stats_kernel");
  if (rc) return rc;
  if (silu) hipLaunchKernelGGL((gn_any_apply_kernel<T, true>), dim3((unsigned)nblk), dim3(GA_NT), 0, s, a);
  else hipLaunchKernelGGL((gn_any_apply_kernel<T, false>), dim3((unsigned)nblk), dim3(GA_NT), 0, s, a);
  return check_launch("gn_any_apply_kernel");
}

// ---------------------------------------------------------------------------------------
// Channels-last, any channels per group.  A thread owns one 16-byte channel vector (column) on
// every R-th position of a chunk; 256 / columns rows of threads, the rest of the 256 idle.  A
// column may span several groups and a group several columns, so the moments are kept per channel:
//   stats: each thread sums its positions of a channel about the mean of its first four, and the
//          threads' (mean, M2) are merged exactly, over the thread rows and then over the group's
//          channels, in a fixed order; one (mean, M2) record per (chunk, group).  A value far
//          from the rest thus cancels against the n positions of its own thread at a quarter of
//          its size, which bounds M2's relative error by about n / 16 * 2^-24 (one shift for a
//          chunk and group let it reach rows * channels * 2^-24: 3e-4 in rstd over
//          [1, 96, 96, 96], G = 1 with one value of 1e3, now 1e-7).
//   apply: every workgroup merges its sample's records itself (the first rows of x are loaded
//          before that), then normalises its chunk.
// [16, 128, 64, 64] bf16 with SiLU: 73.9 us (stock: layout copies, moments, scale, SiLU) -> 13.4 us by
// graph replay: 5.8 the statistics (2.9 TB/s; 6.2 with the chunk-wide shift, whose positions past
// the chunk were computed and masked), 8.8 the second pass (3.8 TB/s; 11.2 when the 16 parameters
// of a thread were loaded one by one after the merge).
// ---------------------------------------------------------------------------------------
constexpr int GC_NT = 256;
constexpr int GC_MAXG = 256;
constexpr int GC_U = 8;  // rows in flight per thread

struct GcArgs {
  const void* x;
  const void* gamma;
  const void* beta;
  void* y;
  float2* part;  // [N][NCH][G]: mean, M2
  int64_t S;
  int N, C, G, cpg, NCH;
  int rows;      // positions per chunk
  int cols, R;   // channel vectors, thread rows
  FastDiv div_r;
  float eps;
  int pdt;
};

// A chunk is one batch of rows in flight per thread (GC_U for every thread row of a 16-bit tensor):
// rounded down, the few rows over a batch cost a second round trip ([1, 128, 37, 53] bf16 11.8 us,
// rounded up 10.5).  A quarter of that where it leaves under 64 workgroups ([16, 96, 17, 19] 10.4
// -> 9.6 us).  At most two workgroups per CU, the 64 records a group that 8 lanes load at once
// ([4, 128, 128, 128] 128 chunks 18.2 us, 64 chunks 15.4), and more only while a CU is without a
// workgroup ([1, 128, 256, 256] 64 chunks 30.1 us, 256 chunks 21.0).
int gc_chunks(int64_t N, int64_t C, int64_t S) {
  const int64_t batch = std::max<int64_t>(1, GC_NT / std::max<int64_t>(1, C / 8)) * GC_U;
  const int64_t n = std::max<int64_t>(1, N);
  int64_t ch = (S + batch - 1) / batch;
  if (n * ch < 64) ch = std::min<int64_t>((S * 4 + batch - 1) / batch, std::max<int64_t>(ch, 64));
  ch = std::max<int64_t>(1, std::min<int64_t>(ch, std::max<int64_t>(256 / n, std::min<int64_t>(512 / n, 64))));
  const int64_t rows = (S + ch - 1) / ch;
  return (int)((S + rows - 1) / rows);
}

// Mean of the first four of p[0], p[stride], .. (n of them; the last stands in for those missing): the
// shift of a merge, such that one far value among them weighs a quarter.
__device__ __forceinline__ float mean4(const float* p, int stride, int n) {
  const float t0 = p[0], t1 = p[min(1, n - 1) * stride], t2 = p[min(2, n - 1) * stride], t3 = p[min(3, n - 1) * stride];
  return 0.25f * ((t0 + t1) + (t2 + t3));
}

template <typename T>
__global__ __launch_bounds__(GC_NT) void gn_cl_any_stats_kernel(GcArgs a, int lanes) {
  constexpr int VEC = Vec16<T>::N;
  __shared__ __align__(16) float l1[GC_NT * VEC], l2[GC_NT * VEC];
  const int tid = threadIdx.x, r = tid / a.cols, v = tid - r * a.cols;
  const int n = blockIdx.x / a.NCH, ch = blockIdx.x - n * a.NCH;
  const int64_t s0 = (int64_t)ch * a.rows, s1 = min(s0 + a.rows, a.S);
  const T* __restrict__ xn = static_cast<const T*>(a.x) + (int64_t)n * a.S * a.C;
  // thread row q holds per + (q < more) of the chunk's len positions
  const int len = (int)(s1 - s0), per = (int)fdiv((uint32_t)len, a.div_r), more = len - per * a.R;
  const float wl = (float)per, wm = (float)(per + 1);
  if (r < a.R) {
    Vec16<T> b[GC_U];
    auto issue = [&](int64_t p0) {
#pragma unroll
      for (int u = 0; u < GC_U; ++u)
        b[u].raw = *reinterpret_cast<const uint4*>(xn + min(p0 + (int64_t)u * a.R, s1 - 1) * a.C + v * VEC);
    };
    float K[VEC], a1[VEC], a2[VEC];
    auto add = [&](int64_t p0) {
      // all of a batch is requested before any of it is used (else it is waited for in turn)
#pragma unroll
      for (int u = 0; u < GC_U; ++u)
        asm volatile("" : : "v"(b[u].raw.x), "v"(b[u].raw.y), "v"(b[u].raw.z), "v"(b[u].raw.w));
#pragma unroll
      for (int u = 0; u < GC_U; ++u) {
        if (p0 + (int64_t)u * a.R >= s1) break;
#pragma unroll
        for (int k = 0; k < VEC; ++k) {
          const float d = to_f32(b[u].e[k]) - K[k];
          a1[k] += d;
          a2[k] = fmaf(d, d, a2[k]);
        }
      }
    };
    int64_t p0 = s0 + r;
    issue(p0);
#pragma unroll
    for (int k = 0; k < VEC; ++k) {  // (positions past the chunk repeat its last one: any value is a shift)
      K[k] = 0.25f * ((to_f32(b[0].e[k]) + to_f32(b[1].e[k])) + (to_f32(b[2].e[k]) + to_f32(b[3].e[k])));
      a1[k] = a2[k] = 0.f;
    }
    add(p0);
    while ((p0 += (int64_t)GC_U * a.R) < s1) {
      issue(p0);
      add(p0);
    }
    const int cnt = per + (r < more);
    const float inv = cnt ? __builtin_amdgcn_rcpf((float)cnt) : 0.f;
    float4* o1 = reinterpret_cast<float4*>(l1 + r * a.C + v * VEC);
    float4* o2 = reinterpret_cast<float4*>(l2 + r * a.C + v * VEC);
#pragma unroll
    for (int k = 0; k < VEC; ++k) {
      const float q = a1[k] * inv;
      a2[k] = fmaxf(fmaf(-a1[k], q, a2[k]), 0.f);
      a1[k] = cnt ? K[k] + q : 0.f;
    }
#pragma unroll
    for (int k = 0; k < VEC; k += 4) {
      o1[k / 4] = make_float4(a1[k], a1[k + 1], a1[k + 2], a1[k + 3]);
      o2[k / 4] = make_float4(a2[k], a2[k + 1], a2[k + 2], a2[k + 3]);
    }
  }
  __syncthreads();
  const float inv_len = __builtin_amdgcn_rcpf((float)len);
  for (int c = 2 * tid; c < a.C; c += 2 * GC_NT) {  // over the thread rows, two channels a thread, into row 0
    const float m0 = mean4(l1 + c, a.C, a.R), n0 = mean4(l1 + c + 1, a.C, a.R);
    float t1 = 0.f, t2 = 0.f, u1 = 0.f, u2 = 0.f;
#pragma unroll 4
    for (int q = 0; q < a.R; ++q) {
      const float2 m = *reinterpret_cast<const float2*>(l1 + q * a.C + c);
      const float2 s = *reinterpret_cast<const float2*>(l2 + q * a.C + c);
      const float w = q < more ? wm : wl, d = m.x - m0, e = m.y - n0;
      t1 = fmaf(w, d, t1);
      u1 = fmaf(w, e, u1);
      t2 += fmaf(w * d, d, s.x);
      u2 += fmaf(w * e, e, s.y);
    }
    const float q = t1 * inv_len, h = u1 * inv_len;
    *reinterpret_cast<float2*>(l1 + c) = make_float2(m0 + q, n0 + h);
    *reinterpret_cast<float2*>(l2 + c) = make_float2(fmaxf(fmaf(-t1, q, t2), 0.f), fmaxf(fmaf(-u1, h, u2), 0.f));
  }
  __syncthreads();
  // `lanes` lanes (a power of two) per group, over its channels
  const int j = tid & (lanes - 1), g = tid / lanes;
  if (g < a.G) {
    const float* gm = l1 + g * a.cpg;
    const float* gq = l2 + g * a.cpg;
    const float m0 = mean4(gm, 1, a.cpg);
    float t1 = 0.f, t2 = 0.f, t3 = 0.f;
#pragma unroll 4
    for (int i = j; i < a.cpg; i += lanes) {
      const float d = gm[i] - m0;
      t1 += d;
      t2 = fmaf(d, d, t2);
      t3 += gq[i];
    }
    for (int o = lanes >> 1; o; o >>= 1) {
      t1 += __shfl_xor(t1, o, 64);
      t2 += __shfl_xor(t2, o, 64);
      t3 += __shfl_xor(t3, o, 64);
    }
    const float q = t1 * __builtin_amdgcn_rcpf((float)a.cpg);
    if (j == 0)
      a.part[((int64_t)n * a.NCH + ch) * a.G + g] =
          make_float2(m0 + q, fmaf((float)len, fmaxf(fmaf(-t1, q, t2), 0.f), t3));
  }
}

template <typename T, bool SILU>
__global__ __launch_bounds__(GC_NT) void gn_cl_any_apply_kernel(GcArgs a, int lanes) {
  constexpr int VEC = Vec16<T>::N;
  __shared__ float g_mean[GC_MAXG], g_rstd[GC_MAXG];
  const int tid = threadIdx.x, r = tid / a.cols, v = tid - r * a.cols;
  const int n = blockIdx.x / a.NCH, ch = blockIdx.x - n * a.NCH;
  const int64_t s0 = (int64_t)ch * a.rows, s1 = min(s0 + a.rows, a.S);
  const T* __restrict__ xn = static_cast<const T*>(a.x) + (int64_t)n * a.S * a.C;
  T* __restrict__ yn = static_cast<T*>(a.y) + (int64_t)n * a.S * a.C;
  Vec16<T> b[GC_U];
  auto issue = [&](int64_t p0) {
#pragma unroll
    for (int u = 0; u < GC_U; ++u) {
      const uint4* p = reinterpret_cast<const uint4*>(xn + min(p0 + (int64_t)u * a.R, s1 - 1) * a.C + v * VEC);
      b[u].raw = ld16<true>(p);  // the last read of x
    }
  };
  float gm[VEC], bt[VEC];
#pragma unroll
  for (int k = 0; k < VEC; ++k) {
    gm[k] = 1.f;
    bt[k] = 0.f;
  }
  if (r < a.R) {
    issue(s0 + r);
    if (a.gamma) load_params<VEC>(a.gamma, a.pdt, v * VEC, 1, gm);
    if (a.beta) load_params<VEC>(a.beta, a.pdt, v * VEC, 1, bt);
  }
  // `lanes` lanes (a power of two, at most 64) per group merge the sample's records in a fixed order
  const int j = tid & (lanes - 1);
  for (int g = tid / lanes; g < a.G; g += GC_NT / lanes) {
    const float2* p = a.part + (int64_t)n * a.NCH * a.G + g;
    auto cnt = [&](int i) { return (float)(min((int64_t)(i + 1) * a.rows, a.S) - (int64_t)i * a.rows); };
    // a lane's records are loaded together (each load waited for in turn costs its full latency)
    constexpr int RB = 8;
    float2 m[RB];
    float sm = 0.f, q = 0.f;
    auto fetch = [&](int i0) {
#pragma unroll
      for (int t = 0; t < RB; ++t) m[t] = p[(int64_t)min(i0 + t * lanes, a.NCH - 1) * a.G];
    };
    for (int i0 = j; i0 < a.NCH; i0 += RB * lanes) {
      fetch(i0);
#pragma unroll
      for (int t = 0; t < RB; ++t) sm += i0 + t * lanes < a.NCH ? cnt(i0 + t * lanes) * m[t].x : 0.f;
    }
    for (int o = lanes >> 1; o; o >>= 1) sm += __shfl_xor(sm, o, 64);
    const float mean = sm / (float)a.S;
    for (int i0 = j; i0 < a.NCH; i0 += RB * lanes) {
      if (a.NCH > RB * lanes) fetch(i0);  // else the records are still there
#pragma unroll
      for (int t = 0; t < RB; ++t) {
        const float d = m[t].x - mean;
        q += i0 + t * lanes < a.NCH ? m[t].y + cnt(i0 + t * lanes) * (float)a.cpg * d * d : 0.f;
      }
    }
    for (int o = lanes >> 1; o; o >>= 1) q += __shfl_xor(q, o, 64);
    if (j == 0) {
      g_mean[g] = mean;
      g_rstd[g] = 1.0f / sqrtf(q / ((float)a.S * (float)a.cpg) + a.eps);
    }
  }
  __syncthreads();
  if (r >= a.R) return;
  float sc[VEC], sh[VEC];
  int g = v * VEC / a.cpg, left = (g + 1) * a.cpg - v * VEC;  // the channel's group, channels left in it
#pragma unroll
  for (int k = 0; k < VEC; ++k) {
    sc[k] = g_rstd[g] * gm[k];
    sh[k] = bt[k] - g_mean[g] * sc[k];
    const bool next = --left == 0;
    g = min(g + next, a.G - 1);
    left = next ? a.cpg : left;
  }
  for (int64_t p0 = s0 + r; p0 < s1; p0 += (int64_t)GC_U * a.R) {
    if (p0 != s0 + r) issue(p0);
#pragma unroll
    for (int u = 0; u < GC_U; ++u) {
      const int64_t p = p0 + (int64_t)u * a.R;
      float o[VEC];
#pragma unroll
      for (int k = 0; k < VEC; ++k) {
        o[k] = fmaf(to_f32(b[u].e[k]), sc[k], sh[k]);
        if constexpr (SILU) o[k] = silu_f32(o[k]);
      }
      if (p < s1) st16<true>(yn + p * a.C + v * VEC, pack16<T>(o));
    }
  }
}

template <typename T>
int launch_cl_any(GcArgs a, int silu, hipStream_t s) {
  a.cols = a.C / (16 / (int)sizeof(T));
  a.R = GC_NT / a.cols;
  a.div_r = make_fastdiv((uint32_t)a.R);
  int lanes = 64;
  while (lanes > 1 && lanes * a.G > GC_NT) lanes >>= 1;
  const dim3 grid((unsigned)((int64_t)a.N * a.NCH));
  // (a few channels are summed faster than lanes are merged)
  hipLaunchKernelGGL((gn_cl_any_stats_kernel<T>), grid, dim3(GC_NT), 0, s, a, a.cpg >= 32 ? lanes : 1);
  const int rc = check_launch("gn_cl_any_stats_kernel");
  if (rc) return rc;
  if (silu) hipLaunchKernelGGL((gn_cl_any_apply_kernel<T, true>), grid, dim3(GC_NT), 0, s, a, lanes);
  else hipLaunchKernelGGL((gn_cl_any_apply_kernel<T, false>), grid, dim3(GC_NT), 0, s, a, lanes);
  return check_launch("gn_cl_any_apply_kernel");
}

}  // namespace

int gn_any_fwd(const void* x, const void* gamma, const void* beta, void* y, int64_t ngroups, int G, int64_t cpg,
               int64_t S, float eps, int silu, int dtype, int pdt, float* partials, int NS, int64_t slice,
               hipStream_t s) {
  if (S < (int64_t)(16 / dtype_size(dtype))) return fail(ATK_UNSUPPORTED, "group_norm: rows under 16 bytes");
  GaArgs a{};
  a.x = x; a.gamma = gamma; a.beta = beta; a.y = y;
  a.E = cpg * S;
  a.S = (uint32_t)S; a.cpg = (uint32_t)cpg; a.G = (uint32_t)G;
  a.eps = eps; a.pdt = pdt;
  a.div_s = make_fastdiv((uint32_t)S);
  a.partials = partials; a.NS = NS; a.slice = slice;
  switch (dtype) {
    case ATK_F32: return launch_any<float>(a, ngroups, silu, s);
    case ATK_F16: return launch_any<_Float16>(a, ngroups, silu, s);
    default: return launch_any<__bf16>(a, ngroups, silu, s);
  }
}

bool gn_cl_any_takes(int64_t C, int G, int dtype) {
  const int64_t vec = (int64_t)(16 / dtype_size(dtype));
  return C % vec == 0 && C / vec <= GC_NT && G <= GC_MAXG;
}

size_t gn_cl_any_workspace_bytes(int64_t N, int64_t C, int64_t S, int G) {
  return (size_t)N * (size_t)gc_chunks(N, C, S) * (size_t)G * sizeof(float2);
}

int gn_cl_any_fwd(const void* x, const void* gamma, const void* beta, void* y, int64_t N, int64_t C, int64_t S, int G,
                  float eps, int silu, int dtype, int pdt, void* workspace, hipStream_t s) {
  GcArgs a{};
  a.x = x; a.gamma = gamma; a.beta = beta; a.y = y;
  a.part = static_cast<float2*>(workspace);
  a.S = S; a.N = (int)N; a.C = (int)C; a.G = G; a.cpg = (int)(C / G);
  a.NCH = gc_chunks(N, C, S);
  a.rows = (int)((S + a.NCH - 1) / a.NCH);
  a.eps = eps; a.pdt = pdt;
  if (N * a.NCH > 0x7fffffff) return fail(ATK_UNSUPPORTED, "group_norm (channels-last): grid too large");
  switch (dtype) {
    case ATK_F32: return launch_cl_any<float>(a, silu, s);
    case ATK_F16: return launch_cl_any<_Float16>(a, silu, s);
    default: return launch_cl_any<__bf16>(a, silu, s);
  }
}

}  // namespace atk
