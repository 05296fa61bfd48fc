// Weight (and bias) gradient of a stride-1 "same" 3x3(x3) conv2d / conv3d on gfx950 MFMA.
//
//   dW[co, ci, kz, ky, kx] = sum_{n, z, y, x} dy[n, co, z, y, x] * x[n, ci, z+kz-pd, y+ky-1, x+kx-1]
//   db[co]                 = sum_{n, z, y, x} dy[n, co, z, y, x]
//
// (x = 0 outside the input).  The reference computes this with aten.convolution_backward
// (amd_tuned_torch/_dispatch.py:2064-2075).  As a GEMM it is M = Co, N = Ci, K = output
// positions, once per tap; any Ci and Co, any spatial size with W >= 8.
//  * Positions are taken in runs of 8 along a row (a row's last run may be partial).  A wave's
//    K step is two runs, one per half wave, so a row costs ceil(W / 8) runs and not a multiple
//    of 16 positions.
//  * A operand (32 co x 16 positions): a lane's run of dy is one 16-byte global load, shared by
//    all 9 in-plane taps.  Rows need no alignment (global loads may be 2-byte aligned).  A
//    partial run is loaded as the row's last 8 elements and shifted down, so that no load
//    leaves the row and the missing positions are zero.
//  * B operand (16 positions x 32 ci): for a workgroup's 32 input channels, TY + 2 input rows of
//    the plane z+kz-pd are staged in LDS from column x0 - 1 on.  For a run at c a lane reads
//    elements [c, c + 10) of the staged row: one b128 and one b32; the kx = 0 and kx = 2
//    fragments are those dwords as they are and kx = 1 is byte-aligned from them (4 v_alignbyte).
//    Staging from x0 itself, as an earlier form did, took a third LDS read and 4 more aligns,
//    and kept the LDS busy for as long as the MFMAs.
//  * A workgroup = 8 waves = WCO x 32 output channels x 32 input channels x one kz, WP = 8 / WCO
//    waves sharing an output-channel block's positions; each wave holds 3x3 accumulator tiles
//    (144 fp32 registers).  The WP waves' sums are added through LDS at the end.  WCO is 4, 2
//    or 1: the largest that leaves at most an eighth of the output channels' blocks empty.
//  * Stages (TY output rows of one plane) are cut into chunks across workgroups, at most one
//    workgroup per CU; each writes its fp32 partials in the accumulator layout (one 1 KB run
//    per store instruction), summed in a fixed order by a reduce kernel (deterministic) that
//    turns them into the weight layout through LDS.  Partials written straight in the weight
//    layout cost more than all the MFMAs.
// The next stage's input rows are loaded into registers while the current stage computes and
// stored into the other LDS buffer before the one barrier of a stage.
//
// MFMA-bound in principle (floor at 1.23 PFLOP/s, a large bf16 GEMM here: 21 us for 128 -> 128
// channels, 8x45x80, k3); what holds it above that is the dy loads, each lane of which touches a
// row of its own, and the partials.  Measured with the reduce and db: that shape 58 us against
// 410 us for aten.convolution_backward (im2col and a GEMM), 64 -> 64 channels on 16x64x64, 3x3 in
// fp16 29 us, of which the partials of 128 chunks are a third; 5x96x12x11x30 -> 192 62 us
// against 298 us.  Before this kernel all of these took aten's backward.
#include <algorithm>
#include <atomic>

#include "conv_common.h"

namespace atk {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int WG_NT = 512;   // 8 waves
constexpr int WG_CI = 32;    // input channels per workgroup
constexpr int WG_LD = 7;     // 16-byte staging loads per thread
constexpr int WG_PF = 4;     // dy runs in flight per lane
constexpr int WG_LDS_MAX = 160 * 1024;
constexpr int WG_UNIT = 9 * 16 * 64;  // partial floats of one wave: 9 taps x 16 registers x 64 lanes
constexpr int WG_RG = 2;              // chunk groups of the reduce kernel
constexpr int WG_RNT = 288 * WG_RG;   // reduce workgroup: (9 taps x 32 input channels) x groups

struct WgArgs {
  const void* x;
  const void* dy;
  float* part;                 // [chunks][kz][nco][nci][tap 9][reg quad 4][lane 64][4]
  float* dbpart;               // [chunks * WP][nco * 32], or null
  void* dw;                    // [Co][Ci][KD*9]
  void* db;                    // [Co], or null
  int N, Ci, Co, D, H, W, KD, pd;
  int nci, nco, ncog;          // 32-channel blocks; output-channel blocks per WCO
  int TY, ty_tiles;            // output rows per stage, stages per plane column
  int TS, tx_tiles;            // columns per stage (a multiple of 8 where tx_tiles > 1)
  int pitch;                   // staged row pitch in elements
  int slab;                    // elements per input channel in LDS (rows * pitch, bank padded)
  int slab_pad;                // slab - rows * pitch
  int runs_row;                // 16-byte chunks per staged row
  int nload;                   // 16-byte chunks per stage
  int stages, spc, chunks;     // a chunk is a run of spc stages
  int zero_off;                // LDS element offset of a zeroed stretch of 2 * pitch + 16 elements
  FastDiv f_tx, f_ty, f_d;
};

template <typename T>
__device__ __forceinline__ void mfma(f32x16& acc, const uint4& a, const uint4& b) {
  if constexpr (__is_same(T, __bf16))
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*reinterpret_cast<const bf16x8*>(&a),
                                                  *reinterpret_cast<const bf16x8*>(&b), acc, 0, 0, 0);
  else
    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(*reinterpret_cast<const f16x8*>(&a),
                                                 *reinterpret_cast<const f16x8*>(&b), acc, 0, 0, 0);
}

// 16 bytes from a 2-byte aligned global address (a single load: unaligned global access).
__device__ __forceinline__ uint4 gload16u(const char* p) {
  uint4 v;
  __builtin_memcpy(&v, p, 16);
  return v;
}

// The 8 elements of `v` moved down by d elements (zeros move in); d = -1 moves up by one.
__device__ __forceinline__ uint4 shift_elems(uint4 v, int d) {
  uint64_t lo = ((uint64_t)v.y << 32) | v.x, hi = ((uint64_t)v.w << 32) | v.z;
  if (d < 0) {
    hi = (hi << 16) | (lo >> 48);
    lo <<= 16;
  } else {
    if (d >= 4) { lo = hi; hi = 0; }
    const int b = 16 * (d & 3);
    lo = (lo >> b) | ((hi << 1) << (63 - b));
    hi >>= b;
  }
  return make_uint4((uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32));
}

// RAG: W is not a multiple of 8 (rows end in a partial run).
template <typename T, int WCO, bool RAG>
__global__ __launch_bounds__(WG_NT) __attribute__((amdgpu_waves_per_eu(2, 2))) void conv_wgrad_kernel(WgArgs a) {
  constexpr int WP = 8 / WCO;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T* s_x = reinterpret_cast<T*>(smem_raw);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wco = wave % WCO, wp = wave / WCO;
  const int col = lane & 31, half = lane >> 5;
  // Consecutive workgroup ids are dispatched to the 8 XCDs in turn.  Each XCD gets a
  // contiguous run of logical tiles instead, so the input-channel blocks that read the same
  // dy rows (and the output-channel blocks that read the same input rows) share one L2.
  const int gx = a.nci * a.ncog;
  const int nwg = gridDim.x;
  int lid = blockIdx.x;
  if ((nwg & 7) == 0) lid = (lid & 7) * (nwg >> 3) + (lid >> 3);
  const int bx = lid % gx, kz = (lid / gx) % a.KD, chunk = lid / (gx * a.KD);
  const int ci_blk = bx % a.nci, co_blk = (bx / a.nci) * WCO + wco;
  // channels past the end read the last channel: their sums are never written out
  const int co = min(co_blk * 32 + col, a.Co - 1);
  const int HW = a.H * a.W;
  const int64_t plane = (int64_t)a.D * HW;  // elements per (n, channel) volume
  const bool want_db = a.dbpart && ci_blk == 0 && kz == a.pd;

  const int buf_elems = WG_CI * a.slab;
  for (int i = tid * 8; i < 2 * a.pitch + 16; i += WG_NT * 8)
    *reinterpret_cast<uint4*>(s_x + a.zero_off + i) = make_uint4(0, 0, 0, 0);

  f32x16 acc[3][3];
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
  float dbsum = 0.f;

  // staging map: chunk q of 16 bytes -> (ci c, staged row r, run j of the row).  goff: its
  // element offset from row 0, column x0 of the stage's first channel; map: c << 16 | r << 8 | j
  const int per_c = (a.TY + 2) * a.runs_row;
  const int c_last = a.Ci - ci_blk * WG_CI - 1;
  int map[WG_LD], goff[WG_LD];
#pragma unroll
  for (int k = 0; k < WG_LD; ++k) {
    const int q = tid + k * WG_NT;
    const int c = q / per_c, rem = q - c * per_c;
    const int r = rem / a.runs_row, j = rem - r * a.runs_row;
    map[k] = (c << 16) | (r << 8) | j;
    goff[k] = min(c, c_last) * (int)plane + j * 8 - 1;
  }

  struct Stage { int n, z, y0, x0; };
  auto decode = [&](int st) {
    Stage s;
    const int t = (int)fdiv((uint32_t)st, a.f_tx);
    s.x0 = (st - t * a.tx_tiles) * a.TS;
    const int pl = (int)fdiv((uint32_t)t, a.f_ty);
    s.y0 = (t - pl * a.ty_tiles) * a.TY;
    s.n = (int)fdiv((uint32_t)pl, a.f_d);
    s.z = pl - s.n * a.D;
    return s;
  };
  // the first stage at or after st whose input plane z + kz - pd exists (else that tap reads
  // only zero padding)
  const int st_end = min((chunk + 1) * a.spc, a.stages);
  auto next_live = [&](int st) {
#pragma clang loop vectorize(disable) unroll(disable)
    for (; st < st_end; ++st) {
      const int zi = decode(st).z + kz - a.pd;
      if (zi >= 0 && zi < a.D) break;
    }
    return st;
  };
  uint4 buf[WG_LD];
  // Element offset of chunk k: rows outside the plane read the nearest row, and a row's ends run
  // into its neighbours (stage_store masks both), so only the tensor's first and last row can
  // leave it.
  const int x_lim = (int)((int64_t)a.N * a.Ci * plane) - 8;
  auto chunk_off = [&](const Stage& s, int k) {
    int m = map[k];
    asm volatile("" : "+v"(m));  // unpacked here and not kept unpacked across the loop
    const int yi = min(max(s.y0 - 1 + ((m >> 8) & 0xff), 0), a.H - 1);
    const int base = (int)(((int64_t)s.n * a.Ci + ci_blk * WG_CI) * plane + (int64_t)(s.z + kz - a.pd) * HW) + s.x0;
    return base + goff[k] + (int)__umul24((uint32_t)yi, (uint32_t)a.W);
  };
  auto stage_load = [&](const Stage& s) {
#pragma unroll
    for (int k = 0; k < WG_LD; ++k) {
      const int off = min(max(chunk_off(s, k), 0), x_lim);
      buf[k] = gload16u(reinterpret_cast<const char*>(a.x) + (uint32_t)off * 2u);
    }
  };
  auto stage_store = [&](const Stage& s, T* dst) {
    const int zi = s.z + kz - a.pd;
    const bool ends = (s.n == 0 && ci_blk == 0 && zi == 0 && s.y0 <= 1) ||
                      (s.n == a.N - 1 && c_last < WG_CI && zi == a.D - 1 && s.y0 + a.TY + 1 >= a.H);
    const bool y_edge = s.y0 == 0 || s.y0 + a.TY + 1 > a.H;
#pragma unroll
    for (int k = 0; k < WG_LD; ++k) {
      uint4 v = buf[k];
      if (ends) {
        const int off = chunk_off(s, k);
        v = shift_elems(v, min(off - min(max(off, 0), x_lim), 7));
      }
      int m = map[k];
      asm volatile("" : "+v"(m));
      const int c = m >> 16, r = (m >> 8) & 0xff, j = m & 0xff;
      // columns -1 and W on are zero padding.  Where W is a multiple of 8 only the first dword of
      // the chunk past the row is ever read, and column W - 1 is its first element.
      v.x &= s.x0 == 0 && j == 0 ? 0xffff0000u : ~0u;
      const int left = a.W - s.x0 + 1 - j * 8;  // elements of the chunk inside the row
      if (!RAG) {
        v.x &= left == 1 ? 0x0000ffffu : ~0u;
      } else if (left < 8) {
        const uint4 keep = shift_elems(make_uint4(~0u, ~0u, ~0u, ~0u), 8 - max(left, 1));
        v.x &= left > 0 ? keep.x : 0u; v.y &= left > 0 ? keep.y : 0u;
        v.z &= left > 0 ? keep.z : 0u; v.w &= left > 0 ? keep.w : 0u;
      }
      if (y_edge) {
        const int yi = s.y0 - 1 + r;
        if (yi < 0 || yi >= a.H) v = make_uint4(0, 0, 0, 0);
      }
      if (tid + k * WG_NT < a.nload) *reinterpret_cast<uint4*>(dst + (tid + k * WG_NT) * 8 + c * a.slab_pad) = v;
    }
  };

  int st = next_live(chunk * a.spc);
  Stage cur = decode(min(st, a.stages - 1));
  int pb = 0;  // LDS buffer of the current stage
  if (st < st_end) {
    stage_load(cur);
    stage_store(cur, s_x);
  }
  __syncthreads();
  const int rem = a.W & 7;
  const int g_lim = (int)((int64_t)a.N * a.Co * plane) - 8;
  while (st < st_end) {
    const int rows = min(a.TY, a.H - cur.y0);
    const int cols = min(a.TS, a.W - cur.x0);
    const int runs = (cols + 7) >> 3;             // runs per row of this stage
    const int total = rows * runs;
    const int last = cur.x0 + runs * 8 > a.W ? runs - 1 : -1;  // the partial run of a row
    // run iterator of this lane: run i = 2 (wp + WP t) + half of the stage, by row and column
    const int i0 = 2 * wp + half, row0 = i0 / runs;
    int it_col = i0 - row0 * runs;
    int it_g = (int)(((int64_t)cur.n * a.Co + co) * plane + (int64_t)cur.z * HW) + (cur.y0 + row0) * a.W + cur.x0 +
               it_col * 8;  // element offset in dy
    int it_l = pb * buf_elems + col * a.slab + row0 * a.pitch + it_col * 8;  // element offset in LDS
    const int step_row = 2 * WP / runs, step_col = 2 * WP - step_row * runs;
    const int g_step = step_row * a.W + step_col * 8, l_step = step_row * a.pitch + step_col * 8;
    const int g_wrap = a.W - runs * 8, l_wrap = a.pitch - runs * 8;
    const int nk = total > 2 * wp ? (total - 2 * wp + 2 * WP - 1) / (2 * WP) : 0;  // K steps of this wave
    const bool last_ok = 2 * (wp + WP * (nk - 1)) + half < total;  // the last step may be half empty
    uint4 ar[WG_PF];
    int ob[WG_PF];  // LDS element offset of the run (a multiple of 8), plus 1 for a partial run
    auto fetch = [&](int u) {
      const bool pr = RAG && it_col == last;
      // runs past the stage's end (fetched, never used) stay inside the tensor
      const int off = min(it_g - (RAG && pr ? 8 - rem : 0), g_lim);
      ar[u] = gload16u(reinterpret_cast<const char*>(a.dy) + (uint32_t)off * 2u);
      ob[u] = it_l + (RAG && pr ? 1 : 0);
      it_col += step_col;
      const bool wrap = it_col >= runs;
      it_col -= wrap ? runs : 0;
      it_g += g_step + (wrap ? g_wrap : 0);
      it_l += l_step + (wrap ? l_wrap : 0);
    };
#pragma unroll
    for (int u = 0; u < WG_PF; ++u) fetch(u);
    // the next stage's input rows are requested after this stage's first dy runs: load
    // counters complete in issue order, so the first MFMAs do not wait for the input rows
    const int st2 = next_live(st + 1);
    const Stage nxt = decode(min(st2, a.stages - 1));
    if (st2 < st_end) stage_load(nxt);
    // dword masks that drop element `rem`, the only staged element a partial run's kx = 0
    // fragment would take from inside the row
    const uint32_t keep = RAG ? ((rem & 1) ? 0x0000ffffu : 0xffff0000u) : 0;
    for (int ks0 = 0; ks0 < nk; ks0 += WG_PF) {
#pragma unroll
      for (int u = 0; u < WG_PF; ++u) {
        if (ks0 + u >= nk) break;
        uint4 av = ar[u];
        const bool pr = RAG && (ob[u] & 1);
        int o = RAG ? ob[u] & ~7 : ob[u];
        fetch(u);
        if (RAG) {
          const uint4 sv = shift_elems(av, 8 - rem);
          av.x = pr ? sv.x : av.x; av.y = pr ? sv.y : av.y;
          av.z = pr ? sv.z : av.z; av.w = pr ? sv.w : av.w;
        }
        const bool valid = last_ok | (ks0 + u != nk - 1);
        av.x = valid ? av.x : 0u; av.y = valid ? av.y : 0u;
        av.z = valid ? av.z : 0u; av.w = valid ? av.w : 0u;
        o = valid ? o : a.zero_off;
        if (want_db) {
          Vec16<T> e;
          e.raw = av;
#pragma unroll
          for (int i = 0; i < 8; ++i) dbsum += to_f32(e.e[i]);
        }
        uint4 m = make_uint4(~0u, ~0u, ~0u, ~0u);
        if (RAG) {
          m.x = pr && (rem >> 1) == 0 ? keep : ~0u;
          m.y = pr && (rem >> 1) == 1 ? keep : ~0u;
          m.z = pr && (rem >> 1) == 2 ? keep : ~0u;
          m.w = pr && (rem >> 1) == 3 ? keep : ~0u;
        }
        const T* p = s_x + o;
#pragma unroll
        for (int ky = 0; ky < 3; ++ky) {
          const uint4 d = *reinterpret_cast<const uint4*>(p + ky * a.pitch);
          const uint32_t d4 = *reinterpret_cast<const uint32_t*>(p + ky * a.pitch + 8);
          uint4 f0 = d, f1, f2;
          if (RAG) { f0.x &= m.x; f0.y &= m.y; f0.z &= m.z; f0.w &= m.w; }
          f1.x = __builtin_amdgcn_alignbyte(d.y, d.x, 2);
          f1.y = __builtin_amdgcn_alignbyte(d.z, d.y, 2);
          f1.z = __builtin_amdgcn_alignbyte(d.w, d.z, 2);
          f1.w = __builtin_amdgcn_alignbyte(d4, d.w, 2);
          f2 = make_uint4(d.y, d.z, d.w, d4);
          mfma<T>(acc[ky][0], av, f0);
          mfma<T>(acc[ky][1], av, f1);
          mfma<T>(acc[ky][2], av, f2);
        }
      }
    }
    if (st2 < st_end) stage_store(nxt, s_x + (pb ^ 1) * buf_elems);
    __syncthreads();
    pb ^= 1;
    st = st2;
    cur = nxt;
  }

  if (want_db && co_blk < a.nco) {
    dbsum += __shfl_xor(dbsum, 32, 64);
    if (half == 0) a.dbpart[((int64_t)chunk * WP + wp) * (a.nco * 32) + co_blk * 32 + col] = dbsum;
  }
  // add the WP waves of an output-channel block in order, one ky at a time: 12 KB per wave
  float* s_f = reinterpret_cast<float*>(smem_raw);
  constexpr int SLOT = 3 * 16 * 64;
  if constexpr (WP > 1) {
#pragma unroll
    for (int ky = 0; ky < 3; ++ky) {
      __syncthreads();
      if (wp > 0) {
        float* d = s_f + ((wp - 1) * WCO + wco) * SLOT + lane * 4;
#pragma unroll
        for (int kx = 0; kx < 3; ++kx)
#pragma unroll
          for (int q = 0; q < 4; ++q)
            *reinterpret_cast<float4*>(d + (kx * 4 + q) * 256) =
                make_float4(acc[ky][kx][4 * q], acc[ky][kx][4 * q + 1], acc[ky][kx][4 * q + 2], acc[ky][kx][4 * q + 3]);
      }
      __syncthreads();
      if (wp == 0) {
        for (int g = 0; g < WP - 1; ++g) {
          const float* d = s_f + (g * WCO + wco) * SLOT + lane * 4;
#pragma unroll
          for (int kx = 0; kx < 3; ++kx)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              const float4 v = *reinterpret_cast<const float4*>(d + (kx * 4 + q) * 256);
              acc[ky][kx][4 * q] += v.x;
              acc[ky][kx][4 * q + 1] += v.y;
              acc[ky][kx][4 * q + 2] += v.z;
              acc[ky][kx][4 * q + 3] += v.w;
            }
        }
      }
    }
  }
  if (wp != 0 || co_blk >= a.nco) return;
  // partials in the accumulator layout: one float4 (4 consecutive accumulator registers)
  // per lane, so a store instruction writes 1 KB contiguous
  const int64_t unit = (((int64_t)chunk * a.KD + kz) * a.nco + co_blk) * a.nci + ci_blk;
  float* dst = a.part + unit * WG_UNIT + lane * 4;
#pragma unroll
  for (int ky = 0; ky < 3; ++ky)
#pragma unroll
    for (int kx = 0; kx < 3; ++kx)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<float4*>(dst + ((ky * 3 + kx) * 4 + q) * 256) =
            make_float4(acc[ky][kx][4 * q], acc[ky][kx][4 * q + 1], acc[ky][kx][4 * q + 2], acc[ky][kx][4 * q + 3]);
}

constexpr int WR_NT = 256;   // 4 waves
constexpr int WR_CO = 128;   // output channels per workgroup (32 per wave)
constexpr int WR_TY = 4;     // output rows per stage
constexpr int WR_R = WR_TY + 2;
constexpr int WR_PAD = 8;    // zero elements left / right of each staged row
constexpr int WR_MAXW = 64;  // staging map: 32 ci x 6 rows x W / 8 chunks over 256 threads x 6 loads
constexpr int WR_LD = 6;     // 16-byte staging loads per thread
constexpr int WR_PF = 4;     // dy fragments in flight per lane

struct WgRowArgs {
  const void* x;
  const void* dy;
  float* part;                 // as WgArgs::part
  int N, Ci, Co, D, H, W, KD, pd;
  int stages_per_chunk, chunks;  // a chunk is a run of (n, z, 4-row) stages
  int pitch;                   // staged row pitch in elements (W + 2*PAD)
  int slab;                    // elements per input channel in LDS (R * pitch, bank padded)
  int chunks16;                // 16-byte chunks per staged stage = WG_CI * R * W / 8
  uint32_t x_bytes, dy_bytes;
};

// The weight gradient alone where rows are whole 16-position K steps and output channels whole
// 128-channel blocks (Co % 128, Ci % 32, W % 16 == 0, W <= 64): two workgroups of 4 waves per CU
// whose barriers do not meet, a stage of 4 whole output rows whose dy offsets are linear in the
// K step, and aligned loads throughout.  256 -> 256 channels, 8x64x64, k3 in bf16: 135 us against
// 153 us for conv_wgrad_kernel, which also sums db in that time (a separate reduction of dy takes
// 7 to 21 us, so with a bias the one kernel is as fast).
template <typename T>
__global__ __launch_bounds__(WR_NT, 2) void conv_wgrad_rows_kernel(WgRowArgs a) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T* s_x = reinterpret_cast<T*>(smem_raw);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int col = lane & 31, half = lane >> 5;
  const int n_ci = a.Ci / WG_CI;
  // Consecutive workgroup ids are dispatched to the 8 XCDs in turn.  Each XCD gets a
  // contiguous run of logical tiles instead, so the input-channel blocks that read the same
  // dy rows (and the output-channel blocks that read the same input rows) share one L2.
  const int gx = gridDim.x, gy = gridDim.y;
  const int nwg = gx * gy * gridDim.z;
  int lid = blockIdx.x + gx * (blockIdx.y + gy * blockIdx.z);
  if ((nwg & 7) == 0) lid = (lid & 7) * (nwg >> 3) + (lid >> 3);
  const int bx = lid % gx, kz = (lid / gx) % gy, chunk = lid / (gx * gy);
  const int ci_base = (bx % n_ci) * WG_CI;
  const int co_base = (bx / n_ci) * WR_CO + wave * 32;
  const int HW = a.H * a.W;
  const int64_t plane_x = (int64_t)a.D * HW;  // elements per (n, channel) volume

  const __amdgpu_buffer_rsrc_t rx = make_rsrc(a.x, a.x_bytes);
  const __amdgpu_buffer_rsrc_t rg = make_rsrc(a.dy, a.dy_bytes);

  // zero the row pads once (never overwritten by the staged data)
  for (int i = tid; i < WG_CI * WR_R * 2; i += WR_NT) {
    const int side = i & 1, row = (i >> 1) % WR_R, c = (i >> 1) / WR_R;
    *reinterpret_cast<uint4*>(s_x + c * a.slab + row * a.pitch + (side ? WR_PAD + a.W : 0)) = make_uint4(0, 0, 0, 0);
  }

  f32x16 acc[3][3];
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  // staging map: chunk q of 16 bytes -> (ci c, row r, x0)
  const int xq = a.W >> 3;  // 16-byte chunks per row
  auto stage_load = [&](int n, int zi, int y0, uint4 (&buf)[WR_LD]) {
#pragma unroll
    for (int k = 0; k < WR_LD; ++k) {
      const int q = tid + k * WR_NT;
      const int c = q / (WR_R * xq), rem = q - c * (WR_R * xq);
      const int r = rem / xq, x0 = (rem - r * xq) * 8;
      const int yi = y0 - 1 + r;
      const bool ok = q < a.chunks16 && zi >= 0 && zi < a.D && yi >= 0 && yi < a.H;
      const int64_t e = ((int64_t)n * a.Ci + ci_base + c) * plane_x + ((int64_t)zi * a.H + yi) * a.W + x0;
      buf[k] = bload16(rx, ok ? (uint32_t)(e * (int64_t)sizeof(T)) : kOOB, 0);
    }
  };
  auto stage_store = [&](const uint4 (&buf)[WR_LD]) {
#pragma unroll
    for (int k = 0; k < WR_LD; ++k) {
      const int q = tid + k * WR_NT;
      if (q < a.chunks16) {
        const int c = q / (WR_R * xq), rem = q - c * (WR_R * xq);
        const int r = rem / xq, x0 = (rem - r * xq) * 8;
        *reinterpret_cast<uint4*>(s_x + c * a.slab + r * a.pitch + WR_PAD + x0) = buf[k];
      }
    }
  };

  const int n_ystages = (a.H + WR_TY - 1) / WR_TY;
  const int ksteps_row = a.W >> 4;
  // LDS read base of this lane: input channel `col`, first 8 output positions of its half
  const T* s_lane = s_x + col * a.slab + half * 8;

  uint4 buf[WR_LD];
  int st = chunk * a.stages_per_chunk;
  const int st_end = min(st + a.stages_per_chunk, a.N * a.D * n_ystages);
  if (st < st_end) {
    const int pl = st / n_ystages, ys = st - (st / n_ystages) * n_ystages;
    stage_load(pl / a.D, pl % a.D + kz - a.pd, ys * WR_TY, buf);
  }
  for (; st < st_end; ++st) {
    const int pl = st / n_ystages, ys = st - pl * n_ystages;
    const int n = pl / a.D, z = pl - n * a.D;
    const int y0 = ys * WR_TY;
    __syncthreads();  // previous stage's reads done
    stage_store(buf);
    __syncthreads();
    const int zi = z + kz - a.pd;
    const bool live = zi >= 0 && zi < a.D;  // else this kz tap reads only zero padding (uniform)
    // a stage covers whole output rows, so k-step ks (16 positions) starts at position
    // y0*W + ks*16 of the plane: the dy offset is linear in ks
    const uint32_t g0 = (uint32_t)((((int64_t)n * a.Co + co_base + col) * plane_x + (int64_t)z * HW +
                                    (int64_t)y0 * a.W + half * 8) * (int64_t)sizeof(T));
    const int rows = min(WR_TY, a.H - y0);
    const int nk = live ? rows * ksteps_row : 0;
    uint4 ar[WR_PF];  // dy fragments stream through a ring, WR_PF k-steps ahead
#pragma unroll
    for (int u = 0; u < WR_PF; ++u) ar[u] = bload16(rg, u < nk ? g0 + (uint32_t)u * 32u : kOOB, 0);
    // the next stage's input rows are requested after this stage's first dy fragments: load
    // counters complete in issue order, so the first MFMAs do not wait for the input rows
    if (st + 1 < st_end) {
      const int pl2 = (st + 1) / n_ystages, ys2 = (st + 1) - pl2 * n_ystages;
      stage_load(pl2 / a.D, pl2 % a.D + kz - a.pd, ys2 * WR_TY, buf);
    }
    if (!live) continue;
    int xs = 0;                   // 16-position column block of the current k-step
    const T* prow = s_lane + WR_PAD;  // staged row ty (+ ky below) of the current k-step
    for (int ks0 = 0; ks0 < nk; ks0 += WR_PF) {
#pragma unroll
      for (int u = 0; u < WR_PF; ++u) {
        const int ks = ks0 + u;
        if (ks >= nk) break;
        const uint4 av = ar[u];
        ar[u] = bload16(rg, ks + WR_PF < nk ? g0 + (uint32_t)(ks + WR_PF) * 32u : kOOB, 0);
#pragma unroll
        for (int ky = 0; ky < 3; ++ky) {
          // staged element index of input x' = x0 - 1 + e is PAD + x0 - 1 + e; read dwords
          // covering [PAD + x0 - 2, PAD + x0 + 10): D3 = b32 at PAD+x0-2, D4..7 = b128 at
          // PAD+x0, D8 = b32 at PAD+x0+8  (x0 = xs*16 + half*8, PAD = 8 keeps them aligned)
          const T* p = prow + ky * a.pitch + xs * 16;
          const uint32_t d3 = *reinterpret_cast<const uint32_t*>(p - 2);
          const uint4 d47 = *reinterpret_cast<const uint4*>(p);
          const uint32_t d8 = *reinterpret_cast<const uint32_t*>(p + 8);
          // kx = 0: elements start at x0 - 1 (odd): bytes 2.. of (d3, d4, ..., d7)
          uint4 f0, f2;
          f0.x = __builtin_amdgcn_alignbyte(d47.x, d3, 2);
          f0.y = __builtin_amdgcn_alignbyte(d47.y, d47.x, 2);
          f0.z = __builtin_amdgcn_alignbyte(d47.z, d47.y, 2);
          f0.w = __builtin_amdgcn_alignbyte(d47.w, d47.z, 2);
          // kx = 2: elements start at x0 + 1
          f2.x = __builtin_amdgcn_alignbyte(d47.y, d47.x, 2);
          f2.y = __builtin_amdgcn_alignbyte(d47.z, d47.y, 2);
          f2.z = __builtin_amdgcn_alignbyte(d47.w, d47.z, 2);
          f2.w = __builtin_amdgcn_alignbyte(d8, d47.w, 2);
          mfma<T>(acc[ky][0], av, f0);
          mfma<T>(acc[ky][1], av, d47);
          mfma<T>(acc[ky][2], av, f2);
        }
        if (++xs == ksteps_row) {
          xs = 0;
          prow += a.pitch;
        }
      }
    }
  }

  // partials in the accumulator layout: one float4 (4 consecutive accumulator registers)
  // per lane, so a store instruction writes 1 KB contiguous
  const int64_t unit = (((int64_t)chunk * a.KD + kz) * (a.Co / 32) + (bx / n_ci) * 4 + wave) * n_ci + bx % n_ci;
  float* dst = a.part + unit * WG_UNIT + lane * 4;
#pragma unroll
  for (int ky = 0; ky < 3; ++ky)
#pragma unroll
    for (int kx = 0; kx < 3; ++kx)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<float4*>(dst + ((ky * 3 + kx) * 4 + q) * 256) =
            make_float4(acc[ky][kx][4 * q], acc[ky][kx][4 * q + 1], acc[ky][kx][4 * q + 2], acc[ky][kx][4 * q + 3]);
}

// Sums the chunks' partials in a fixed order and writes dW (and db).  In a wave's accumulator,
// register r = 4 q + e of lane (half, col) holds output channel 8 q + 4 half + e and input
// channel col, so a (q, half) slice is 4 consecutive output channels x 32 input channels: a
// workgroup takes one such slice over every kz and tap, sums it into LDS as
// [co 4][ci 32][kz][tap] -- 4 contiguous runs of dW -- and writes those out.  Each of WG_RG
// thread groups sums every WG_RG-th chunk with 8 loads in flight (a thread that waited for its
// loads in turn was bound by their latency where few blocks share many chunks).  The workgroups
// past the slices sum db, 32 channels each.
template <int KD, typename OT>
__global__ __launch_bounds__(WG_RNT) void conv_wgrad_reduce_kernel(WgArgs a, int db_rows) {
  __shared__ __align__(16) float s_w[WG_RG * 4 * WG_CI * KD * 9];
  constexpr int ROW = WG_CI * KD * 9;  // floats of one output channel's run in dW
  const int t = threadIdx.x;
  const int slices = a.nco * a.nci * 8;
  if ((int)blockIdx.x >= slices) {
    const int co = ((int)blockIdx.x - slices) * 32 + (t & 31), g = t >> 5;
    constexpr int NG = WG_RNT / 32;
    float s = 0.f;
    for (int r = g; r < db_rows; r += NG) s += a.dbpart[(int64_t)r * (a.nco * 32) + co];
    s_w[g * 32 + (t & 31)] = s;
    __syncthreads();
    if (t < 32 && co < a.Co) {
      s = 0.f;
      for (int i = 0; i < NG; ++i) s += s_w[i * 32 + t];
      static_cast<OT*>(a.db)[co] = from_f32<OT>(s);
    }
    return;
  }
  const int half = blockIdx.x & 1, q = (blockIdx.x >> 1) & 3;
  const int tile = blockIdx.x >> 3;
  const int co_blk = tile / a.nci, ci_blk = tile - co_blk * a.nci;
  const int64_t total = (int64_t)KD * a.nco * a.nci * WG_UNIT;  // partial floats of a chunk
  const int grp = t / 288, tt = t - grp * 288;
  const int tap = tt >> 5, col = tt & 31;
  const int64_t lane_off = (((int64_t)tap * 4 + q) * 64 + half * 32 + col) * 4;
#pragma unroll
  for (int kz = 0; kz < KD; ++kz) {
    const int64_t unit = ((int64_t)kz * a.nco + co_blk) * a.nci + ci_blk;
    const float* src = a.part + unit * WG_UNIT + lane_off;
    float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int c = grp; c < a.chunks; c += 8 * WG_RG) {
      float4 v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int cc = c + u * WG_RG;
        v[u] = *reinterpret_cast<const float4*>(src + (int64_t)min(cc, a.chunks - 1) * total);
        if (cc >= a.chunks) v[u] = make_float4(0.f, 0.f, 0.f, 0.f);
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) { s.x += v[u].x; s.y += v[u].y; s.z += v[u].z; s.w += v[u].w; }
    }
    float* d = s_w + grp * 4 * ROW + col * (KD * 9) + kz * 9 + tap;
    d[0] = s.x;
    d[ROW] = s.y;
    d[2 * ROW] = s.z;
    d[3 * ROW] = s.w;
  }
  __syncthreads();
  const int co0 = co_blk * 32 + q * 8 + half * 4, ci0 = ci_blk * WG_CI;
  const int run = min(WG_CI, a.Ci - ci0) * (KD * 9);
  OT* out = static_cast<OT*>(a.dw) + ((int64_t)co0 * a.Ci + ci0) * (KD * 9);
  for (int i = t; i < 4 * ROW; i += WG_RNT) {
    const int row = i / ROW, e = i - row * ROW;
    if (e < run && co0 + row < a.Co) {
      float v = s_w[i];
#pragma unroll
      for (int g = 1; g < WG_RG; ++g) v += s_w[g * 4 * ROW + i];
      out[(int64_t)row * a.Ci * (KD * 9) + e] = from_f32<OT>(v);
    }
  }
}

int pick_wco(int nco) {
  for (int w = 4; w > 1; w >>= 1) {
    const int padded = (nco + w - 1) / w * w;
    if ((padded - nco) * 8 <= padded) return w;
  }
  return 1;
}

// LDS elements of a stage's rows; the per-channel stride is an odd number of 16-byte units, so
// that a b128 read across channels meets every bank.
int slab_elems(int TY, int runs_row) {
  int units = (TY + 2) * runs_row;
  if (!(units & 1)) ++units;
  return units * 8;
}

void wgrad_plan(int64_t N, int64_t Ci, int64_t Co, int64_t D, int64_t H, int64_t W, int KD, WgArgs* a, int* wco) {
  a->N = (int)N; a->Ci = (int)Ci; a->Co = (int)Co; a->D = (int)D; a->H = (int)H; a->W = (int)W;
  a->KD = KD; a->pd = (KD - 1) / 2;
  a->nci = (int)((Ci + WG_CI - 1) / WG_CI);
  a->nco = (int)((Co + 31) / 32);
  *wco = pick_wco(a->nco);
  const int wp = 8 / *wco;
  a->ncog = (a->nco + *wco - 1) / *wco;
  const int64_t groups = (int64_t)a->nci * a->ncog * KD;
  // Columns per stage: the fewest equal tiles of at most 96 columns.  Rows per stage and chunks:
  // the least estimate of a workgroup's time, in K steps of its busiest wave (9 MFMAs, 288
  // cycles, on a SIMD that two waves share): the steps of its stages, about 2 per stage for the
  // staging (more rows per stage amortise the two halo rows), and 16 for its partials.  At most
  // one workgroup per CU: every workgroup writes up to 147 KB of partials.
  a->tx_tiles = (int)((W + 95) / 96);
  a->TS = (int)((W + a->tx_tiles - 1) / a->tx_tiles + 7) / 8 * 8;
  if (a->tx_tiles > 1) a->tx_tiles = (int)((W + a->TS - 1) / a->TS);
  const int runs = a->TS / 8;
  a->runs_row = runs + 1;
  double best = 0;
  for (int ty = 1; ty <= 16; ++ty) {
    if (WG_CI * (ty + 2) * a->runs_row > WG_LD * WG_NT && ty > 1) break;
    const int64_t tiles = (H + ty - 1) / ty;
    if (ty > 1 && (H + ty - 2) / (ty - 1) == tiles) continue;  // taller, but no fewer stages
    const int64_t stages = N * D * tiles * a->tx_tiles;
    const int64_t most = std::max<int64_t>(1, std::min<int64_t>(256 / groups, stages));
    const int64_t spc = (stages + most - 1) / most, chunks = (stages + spc - 1) / spc;
    const int64_t rounds = (groups * chunks + 255) / 256;
    const double steps = (ty * runs + 2 * wp - 1) / (2 * wp);
    const double cost = (double)rounds * (spc * (2 * steps + 2 + 0.25 * (ty + 2) * runs / 8) + 16) + 0.1 * chunks;
    if (best == 0 || cost < best) {
      best = cost;
      a->TY = ty;
      a->ty_tiles = (int)tiles;
      a->stages = (int)stages;
      a->spc = (int)spc;
      a->chunks = (int)chunks;
    }
  }
  a->pitch = a->runs_row * 8;
  a->slab = slab_elems(a->TY, a->runs_row);
  a->slab_pad = a->slab - (a->TY + 2) * a->pitch;
  a->nload = WG_CI * (a->TY + 2) * a->runs_row;
  a->zero_off = 2 * WG_CI * a->slab;
  a->f_tx = make_fastdiv((uint32_t)a->tx_tiles);
  a->f_ty = make_fastdiv((uint32_t)a->ty_tiles);
  a->f_d = make_fastdiv((uint32_t)D);
}

void rows_plan(int64_t N, int64_t Ci, int64_t Co, int64_t D, int64_t H, int64_t W, int KD, WgRowArgs* a) {
  a->N = (int)N; a->Ci = (int)Ci; a->Co = (int)Co; a->D = (int)D; a->H = (int)H; a->W = (int)W;
  a->KD = KD; a->pd = (KD - 1) / 2;
  a->pitch = (int)W + 2 * WR_PAD;
  int slab = WR_R * a->pitch;               // elements; keep the per-channel stride off a multiple
  while (((slab / 2) & 31) != 4) slab += 8;  // of the bank count (ds_read_b128 across 32 channels)
  a->slab = slab;
  a->chunks16 = (int)(WG_CI * WR_R * (W / 8));
  const int64_t groups = std::max<int64_t>(1, (Ci / WG_CI) * (Co / WR_CO) * KD);
  // as many chunks as keep the grid within one round of 512 resident workgroups (2 per CU):
  // a grid just over a multiple of 512 leaves most CUs idle for its last round.  A chunk
  // spans at least 4 stages, so a workgroup's partials (128 x 32 x 9 floats, 147 KB) stay
  // below half of what it reads (88 KB of input and dy rows per stage at W = 64).
  const int64_t stages = N * D * ((H + WR_TY - 1) / WR_TY);
  int64_t chunks = std::max<int64_t>(1, std::min<int64_t>(512 / groups, stages / 4));
  a->stages_per_chunk = (int)((stages + chunks - 1) / chunks);
  a->chunks = (int)((stages + a->stages_per_chunk - 1) / a->stages_per_chunk);
}

size_t part_floats(const WgArgs& a) { return (size_t)a.chunks * a.KD * a.nco * a.nci * WG_UNIT; }

// Shapes of the kernel: 32-bit offsets inside one tensor, rows of at least one run.
bool wgrad_takes(int64_t N, int64_t Ci, int64_t Co, int64_t D, int64_t H, int64_t W, int KD) {
  if (N <= 0 || Ci <= 0 || Co <= 0 || D <= 0 || H <= 0 || W < 8 || (KD != 1 && KD != 3)) return false;
  const int64_t lim = (int64_t)1 << 30;  // elements: 2 GiB of a 16-bit type
  const int64_t s[] = {N, D, H, W};
  int64_t pos = 1;
  for (int64_t v : s) {
    if (v >= lim || pos >= lim) return false;
    pos *= v;
  }
  // (rows and columns within the 24 bits of chunk_off's product)
  return H < (1 << 24) && W < (1 << 24) && pos < lim && Ci < lim && Co < lim && pos * Ci < lim && pos * Co < lim &&
         Ci * Co < lim / 27;
}

// Shapes of conv_wgrad_rows_kernel, and the limits of atk_conv_wgrad.
bool rows_takes(int64_t Ci, int64_t Co, int64_t W) {
  return Ci % WG_CI == 0 && Co % WR_CO == 0 && W % 16 == 0 && W <= WR_MAXW;
}

size_t workspace_bytes(int64_t N, int64_t Ci, int64_t Co, int64_t D, int64_t H, int64_t W, int KD) {
  WgArgs a{};
  int wco;
  wgrad_plan(N, Ci, Co, D, H, W, KD, &a, &wco);
  size_t floats = part_floats(a) + (size_t)a.chunks * (8 / wco) * a.nco * 32;
  if (rows_takes(Ci, Co, W)) {
    WgRowArgs r{};
    rows_plan(N, Ci, Co, D, H, W, KD, &r);
    floats = std::max(floats, (size_t)r.chunks * Co * Ci * KD * 9);
  }
  return floats * sizeof(float);
}

// The kernels use more than the default 64 KB of dynamic LDS.
template <typename T, int WCO, bool RAG>
int launch_main(const WgArgs& a, dim3 grid, size_t lds, hipStream_t s) {
  if (lds > 64 * 1024) {  // raised once per kernel and device
    static std::atomic<uint64_t> raised{0};
    int dev = 0;
    const uint64_t bit = hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < 64 ? 1ull << dev : 0;
    if (!(raised.load(std::memory_order_relaxed) & bit)) {
      const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&conv_wgrad_kernel<T, WCO, RAG>),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, WG_LDS_MAX);
      if (e != hipSuccess) return fail(ATK_ELAUNCH, "conv_wgrad: cannot raise the LDS limit (%s)", hipGetErrorString(e));
      raised.fetch_or(bit, std::memory_order_relaxed);
    }
  }
  hipLaunchKernelGGL((conv_wgrad_kernel<T, WCO, RAG>), grid, dim3(WG_NT), lds, s, a);
  return check_launch("conv_wgrad_kernel");
}

template <typename T>
int launch_typed(const WgArgs& a, int wco, dim3 grid, size_t lds, hipStream_t s) {
  if (a.W & 7)
    return wco == 4 ? launch_main<T, 4, true>(a, grid, lds, s)
                    : wco == 2 ? launch_main<T, 2, true>(a, grid, lds, s) : launch_main<T, 1, true>(a, grid, lds, s);
  return wco == 4 ? launch_main<T, 4, false>(a, grid, lds, s)
                  : wco == 2 ? launch_main<T, 2, false>(a, grid, lds, s) : launch_main<T, 1, false>(a, grid, lds, s);
}

template <typename OT>
void launch_reduce(const WgArgs& a, int db_rows, hipStream_t s) {
  const dim3 grid((unsigned)(a.nco * a.nci * 8 + (a.db ? a.nco : 0)));
  if (a.KD == 3) hipLaunchKernelGGL((conv_wgrad_reduce_kernel<3, OT>), grid, dim3(WG_RNT), 0, s, a, db_rows);
  else hipLaunchKernelGGL((conv_wgrad_reduce_kernel<1, OT>), grid, dim3(WG_RNT), 0, s, a, db_rows);
}

int reduce_typed(const WgArgs& a, int out_dtype, int db_rows, hipStream_t s) {
  if (out_dtype == ATK_F32) launch_reduce<float>(a, db_rows, s);
  else if (out_dtype == ATK_BF16) launch_reduce<__bf16>(a, db_rows, s);
  else launch_reduce<_Float16>(a, db_rows, s);
  return check_launch("conv_wgrad_reduce_kernel");
}

int run_wgrad(const void* x, const void* dy, void* dw, void* db, int64_t N, int64_t Ci, int64_t D, int64_t H,
              int64_t W, int64_t Co, int KD, int dtype, int out_dtype, void* workspace, size_t ws_bytes,
              hipStream_t s) {
  WgArgs a{};
  int wco;
  wgrad_plan(N, Ci, Co, D, H, W, KD, &a, &wco);
  const int wp = 8 / wco;
  const size_t need = workspace_bytes(N, Ci, Co, D, H, W, KD);
  if (!workspace || ws_bytes < need || (reinterpret_cast<uintptr_t>(workspace) & 15u))
    return fail(ATK_EINVAL, "conv_wgrad: workspace too small or misaligned");
  if (!db && rows_takes(Ci, Co, W) && aligned16(x) && aligned16(dy)) {
    WgRowArgs r{};
    rows_plan(N, Ci, Co, D, H, W, KD, &r);
    r.x = x; r.dy = dy; r.part = static_cast<float*>(workspace);
    r.x_bytes = (uint32_t)(N * Ci * D * H * W * 2);
    r.dy_bytes = (uint32_t)(N * Co * D * H * W * 2);
    const dim3 grid((unsigned)((Ci / WG_CI) * (Co / WR_CO)), (unsigned)KD, (unsigned)r.chunks);
    const size_t lds = (size_t)WG_CI * r.slab * 2;
    if (dtype == ATK_BF16) hipLaunchKernelGGL((conv_wgrad_rows_kernel<__bf16>), grid, dim3(WR_NT), lds, s, r);
    else hipLaunchKernelGGL((conv_wgrad_rows_kernel<_Float16>), grid, dim3(WR_NT), lds, s, r);
    const int rc = check_launch("conv_wgrad_rows_kernel");
    if (rc != ATK_OK) return rc;
    a.chunks = r.chunks;
    a.dw = dw; a.part = r.part;
    return reduce_typed(a, out_dtype, 0, s);
  }
  if (a.nload > WG_LD * WG_NT) return fail(ATK_UNSUPPORTED, "conv_wgrad: staging map too small for W");
  a.x = x; a.dy = dy; a.dw = dw; a.db = db;
  a.part = static_cast<float*>(workspace);
  a.dbpart = db ? a.part + part_floats(a) : nullptr;
  const size_t stage_lds = ((size_t)a.zero_off + 2 * a.pitch + 16) * 2;
  const size_t red_lds = (size_t)(wp - 1) * wco * 3 * 16 * 64 * sizeof(float);
  const size_t lds = std::max(stage_lds, red_lds);
  if (lds > (size_t)WG_LDS_MAX) return fail(ATK_UNSUPPORTED, "conv_wgrad: LDS stage too large");
  const dim3 grid((unsigned)((int64_t)a.nci * a.ncog * KD * a.chunks));
  const int rc = dtype == ATK_BF16 ? launch_typed<__bf16>(a, wco, grid, lds, s)
                                   : launch_typed<_Float16>(a, wco, grid, lds, s);
  if (rc != ATK_OK) return rc;
  return reduce_typed(a, out_dtype, a.chunks * wp, s);
}

}  // namespace
}  // namespace atk

extern "C" size_t atk_conv_wgrad_workspace_bytes(int64_t N, int64_t Ci, int64_t D, int64_t H, int64_t W, int64_t Co,
                                                 int KD) {
  using namespace atk;
  if (!wgrad_takes(N, Ci, Co, D, H, W, KD) || !rows_takes(Ci, Co, W)) return 0;
  return workspace_bytes(N, Ci, Co, D, H, W, KD);
}

extern "C" int atk_conv_wgrad(const void* x, const void* dy, float* dw, int64_t N, int64_t Ci, int64_t D, int64_t H,
                              int64_t W, int64_t Co, int KD, int dtype, void* workspace, size_t ws_bytes,
                              atk_stream_t stream) {
  using namespace atk;
  if (!x || !dy || !dw) return fail(ATK_EINVAL, "conv_wgrad: null pointer");
  if (dtype != ATK_F16 && dtype != ATK_BF16) return fail(ATK_UNSUPPORTED, "conv_wgrad: 16-bit types only");
  if (N <= 0 || Ci <= 0 || Co <= 0 || D <= 0 || H <= 0 || W <= 0) return fail(ATK_EINVAL, "conv_wgrad: bad sizes");
  if (KD != 1 && KD != 3) return fail(ATK_UNSUPPORTED, "conv_wgrad: kernel depth 1 or 3");
  if (!rows_takes(Ci, Co, W))
    return fail(ATK_UNSUPPORTED, "conv_wgrad: needs Ci %% 32, Co %% 128, W %% 16 == 0 and W <= 64");
  if (!aligned16(x) || !aligned16(dy) || !aligned16(dw)) return fail(ATK_UNSUPPORTED, "conv_wgrad: 16-byte aligned tensors");
  if (!wgrad_takes(N, Ci, Co, D, H, W, KD)) return fail(ATK_UNSUPPORTED, "conv_wgrad: tensors over 2 GiB");
  return run_wgrad(x, dy, dw, nullptr, N, Ci, D, H, W, Co, KD, dtype, ATK_F32, workspace, ws_bytes,
                   static_cast<hipStream_t>(stream));
}

extern "C" size_t atk_conv_param_grads_workspace_bytes(int64_t N, int64_t Ci, int64_t D, int64_t H, int64_t W,
                                                       int64_t Co, int KD) {
  using namespace atk;
  return wgrad_takes(N, Ci, Co, D, H, W, KD) ? workspace_bytes(N, Ci, Co, D, H, W, KD) : 0;
}

extern "C" int atk_conv_param_grads(const void* x, const void* dy, void* dw, void* db, int64_t N, int64_t Ci,
                                    int64_t D, int64_t H, int64_t W, int64_t Co, int KD, int dtype, int out_dtype,
                                    void* workspace, size_t ws_bytes, atk_stream_t stream) {
  using namespace atk;
  if (!x || !dy || !dw) return fail(ATK_EINVAL, "conv_param_grads: null pointer");
  if (dtype != ATK_F16 && dtype != ATK_BF16) return fail(ATK_UNSUPPORTED, "conv_param_grads: 16-bit types only");
  if (out_dtype != ATK_F32 && out_dtype != dtype)
    return fail(ATK_UNSUPPORTED, "conv_param_grads: gradients in fp32 or in the input type");
  if (N <= 0 || Ci <= 0 || Co <= 0 || D <= 0 || H <= 0 || W <= 0) return fail(ATK_EINVAL, "conv_param_grads: bad sizes");
  if (!wgrad_takes(N, Ci, Co, D, H, W, KD))
    return fail(ATK_UNSUPPORTED, "conv_param_grads: needs kernel depth 1 or 3, W >= 8 and tensors under 2 GiB");
  if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(dy)) & 1u)
    return fail(ATK_EINVAL, "conv_param_grads: misaligned tensors");
  return run_wgrad(x, dy, dw, db, N, Ci, D, H, W, Co, KD, dtype, out_dtype, workspace, ws_bytes,
                   static_cast<hipStream_t>(stream));
}
