// FullyConnected over ringed uint8 weights: the matmuls of a decode step with a cache as their weights.
//
// The ring over the output channels (query x key cache) is fc_w8_ring_o_kernel, at the end.  The ring over
// the input channels (ConvRuntimeCheckDesc::ring_i_offset_index over a kOSpatialIOGroupI4O4 buffer,
// common/kernels/fully_connected.cc:424-441, 676-706: attention probabilities x value cache) has a long
// window and a narrow output.
//
// The reference's kernel walks the source slices and gathers, for source channel c, the word of
// ring channel (c + offset) % ring_size: four 4-byte reads per slice and output slice.  Here the
// walk is over the ring's own K-slice rows instead: a row (4 ring channels x all output channels)
// is contiguous and aligned, so a thread reads its 16-byte block (4 ring channels x 4 output
// channels) with one load, and what shifts with the offset is the index of the activations:
// row w of the window (w = 0 .. rows touched) is buffer row (offset / 4 + w) % rows and holds
// source channels 4 w - offset % 4 + {0, 1, 2, 3}; those outside [0, channels multiplied) count as
// zero.  That needs ring_size % 4 == 0.
//
// Two kernels walk it: fc_w8_ring_i_column_kernel (one launch; below) and, for the longest windows and wide caches
// at up to 4 tokens, fc_w8_ring_i_kernel, described here.
// Work-group = 256 threads = LS lanes along the output slices x 256 / LS rows in flight, four
// rows per thread and pass; the window is split across blockIdx.x, the slices (in chunks of LS)
// across blockIdx.y, the dst rows of a launch with batched weights across blockIdx.z.  Every
// thread keeps sum(a * (u - 128)) per token and output channel and sum(a) per token; a work-group
// adds its rows through LDS and writes fp32 partial sums to the op's workspace, a second kernel
// adds the parts in their order (fixed), applies scale * (sum - zp * sum(a)), converts and adds
// the bias in the destination type.  MT = token slots per row (1, 2 or 4).
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "kernels.h"

namespace mldhip {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kRingThreads = 256;
// window rows per thread and pass, all of their loads in flight at once: 8 at one token, 4 at more
// (the activations of a row are 8 values per token)
__host__ __device__ constexpr int RingUnroll(int token_slots) { return token_slots == 1 ? 8 : 4; }
constexpr int kRingMaxParts = 256;

struct RingParams {
  const void* act;
  const u32x4* weights;
  const void* scale;
  const void* zero_point;
  const void* bias;
  void* dst;
  float* partial;  // [part][row][token][ns * 4 + 4]: the sums, then sum(a)
  const int32_t* params;
  const int32_t* batch_ids;
  int m, ks, ns;
  int ring_rows;  // ring_size / 4
  int ring_size, ring_index, src_end_ch_index, dst_end_ch_index, k_channels;
  int rows, src_rows, weights_batch;
  int scale_kind, has_zero_point;
  float scalar_scale, scalar_zero_point;
  int parts;
  int xcd_mask, xcd_runs;  // column kernel
};

__device__ __forceinline__ float LoadF(const float* p, size_t i) { return p[i]; }
__device__ __forceinline__ float LoadF(const __half* p, size_t i) { return __half2float(p[i]); }
__device__ __forceinline__ void Load4(const float* p, size_t i, float v[4]) {
  const float4 r = *reinterpret_cast<const float4*>(p + i);
  v[0] = r.x; v[1] = r.y; v[2] = r.z; v[3] = r.w;
}
__device__ __forceinline__ void Load4(const __half* p, size_t i, float v[4]) {
  const uint2 r = *reinterpret_cast<const uint2*>(p + i);
  const __half2 lo = *reinterpret_cast<const __half2*>(&r.x), hi = *reinterpret_cast<const __half2*>(&r.y);
  v[0] = __low2float(lo); v[1] = __high2float(lo); v[2] = __low2float(hi); v[3] = __high2float(hi);
}

// source slices the launch multiplies and dst slices it writes (the runtime channel bounds of the
// unspecialised kernel: fully_connected.cc:750-755, 795)
__device__ __forceinline__ int RingSrcEndSlices(const RingParams& p) {
  if (p.src_end_ch_index < 0) return p.ks;
  return min(max(SrcEndSlices(p.params[p.src_end_ch_index], p.k_channels, p.ks), 0), p.ks);
}
__device__ __forceinline__ int RingDstEndSlice(const RingParams& p) {
  if (p.dst_end_ch_index < 0) return p.ns;
  return min(max(DstEndSlice(p.params[p.dst_end_ch_index], p.ns), 0), p.ns);
}

// sum_i a_i (u_i - 128 - z) for dst channel n of token `token` in row `row`, one product after the other.  The kernels sum
// a_i (u_i - 128) and a_i apart and subtract z times the latter, which turns infinite activations into NaN (without a
// zero point too: -0 * inf); the rare sum of that kind is done over here, as the unspecialised kernel does all of them.
// The arguments are read again from where the kernel got them: kept for this, they would hold 20 scalar registers
// through the whole kernel (and a quarter of the column kernel's speed: one work-group less per CU).
__device__ __forceinline__ bool RingSumInfinite(float asum) { return __builtin_expect(!(fabsf(asum) <= 3.4028235e38f), 0); }
template <typename T, bool RING_O>
__device__ __forceinline__ float RingSumByProducts(int row, int token, int n, float z) {
  typedef const __attribute__((address_space(4))) RingParams* args_t;
  args_t p = (args_t)__builtin_amdgcn_kernarg_segment_ptr();  // (RingParams is each kernel's first argument)
  asm volatile("" : "+s"(p) : : "memory");
  const int ring = p->ring_size, ring_start = ((p->params[p->ring_index] % ring) + ring) % ring;
  int slices = p->ks;
  if (p->src_end_ch_index >= 0) slices = SrcEndSlices(p->params[p->src_end_ch_index], p->k_channels, slices);
  int wb = p->batch_ids ? p->batch_ids[row] : 0;
  wb = min(max(wb, 0), p->weights_batch - 1);
  const T* act = static_cast<const T*>(p->act) + ((size_t)min(row, p->src_rows - 1) * p->m + token) * 4;
  const uint32_t* w32 = reinterpret_cast<const uint32_t*>(p->weights) +
                        (RING_O ? (size_t)wb * p->ks * ring : ((size_t)wb * p->ring_rows * p->ns + (n >> 2)) * 4);
  uint32_t at = ((uint32_t)ring_start + (RING_O ? (uint32_t)n : 0u)) % (uint32_t)ring;  // ring channel
  float sum = 0.0f;
  for (int ks = 0; ks < slices; ++ks) {
    for (int i = 0; i < 4; ++i) {
      const uint32_t word = RING_O ? w32[(size_t)ks * ring + at] : w32[(size_t)(at >> 2) * p->ns * 4 + (at & 3)];
      const float u = (float)((word >> (8 * (RING_O ? i : n & 3))) & 0xFFu);
      sum = fmaf(LoadF(act, (size_t)ks * p->src_rows * p->m * 4 + i), u - (128.0f + z), sum);
      if (!RING_O) at = at + 1 == (uint32_t)ring ? 0u : at + 1;
    }
  }
  return sum;
}

template <typename T, int LS, int MT>
__global__ __launch_bounds__(kRingThreads) void fc_w8_ring_i_kernel(RingParams p) {
  constexpr int RW = kRingThreads / LS;  // window rows in flight per pass
  constexpr int U = RingUnroll(MT);
  __shared__ float red[RW][LS][5 * MT];
  const int tid = threadIdx.x;
  const int s_lane = tid % LS, rsub = tid / LS;
  const int ds = blockIdx.y * LS + s_lane;
  const int row = blockIdx.z;
  int wb = p.batch_ids ? p.batch_ids[row] : 0;
  wb = min(max(wb, 0), p.weights_batch - 1);
  const size_t act_stride = (size_t)p.src_rows * p.m;
  const size_t act_tok0 = (size_t)min(row, p.src_rows - 1) * p.m;
  const T* act = static_cast<const T*>(p.act);
  const int off = ((p.params[p.ring_index] % p.ring_size) + p.ring_size) % p.ring_size;
  const int sh = off & 3, row0 = off >> 2;
  const int ks_end = RingSrcEndSlices(p);
  const int k_eff = ks_end * 4;                      // source channels multiplied (whole slices)
  const int nrows = k_eff > 0 ? (sh + k_eff + 3) >> 2 : 0;  // window rows touched (at most ring_rows + 1)
  const int per = (nrows + p.parts - 1) / p.parts;
  const int w_begin = blockIdx.x * per, w_end = min(nrows, w_begin + per);
  const bool slice_ok = ds < RingDstEndSlice(p);
  const u32x4* wcol = p.weights + (size_t)wb * p.ring_rows * p.ns + min(ds, p.ns - 1);

  float acc[MT][4], asum[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    asum[t] = 0.0f;
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[t][c] = 0.0f;
  }
  for (int w0 = w_begin + rsub; w0 < w_end; w0 += RW * U) {
    u32x4 blk[U];
    float a[U][MT][8];  // [row][token]: source slices w - 1 and w of the window row
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int w = w0 + u * RW;
      const bool live = w < w_end;
      int kb = row0 + min(w, w_end - 1);
      if (kb >= p.ring_rows) kb -= p.ring_rows;
      blk[u] = __builtin_nontemporal_load(wcol + (size_t)kb * p.ns);
      if (!live) blk[u] = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        const bool tok = live && t < p.m;
        // slice w holds source channels 4 w .. 4 w + 3; the row needs 4 w - sh .. 4 w - sh + 3
        const bool lo_ok = tok && sh > 0 && w >= 1 && w - 1 < ks_end, hi_ok = tok && w < ks_end;
        const size_t tk = act_tok0 + min(t, p.m - 1);
        Load4(act, ((size_t)max(min(w - 1, ks_end - 1), 0) * act_stride + tk) * 4, &a[u][t][0]);
        Load4(act, ((size_t)max(min(w, ks_end - 1), 0) * act_stride + tk) * 4, &a[u][t][4]);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          a[u][t][i] = lo_ok ? a[u][t][i] : 0.0f;
          a[u][t][4 + i] = hi_ok ? a[u][t][4 + i] : 0.0f;
        }
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t word = blk[u][i];
        const float u0 = (float)(word & 0xFFu) - 128.0f, u1 = (float)((word >> 8) & 0xFFu) - 128.0f;
        const float u2 = (float)((word >> 16) & 0xFFu) - 128.0f, u3 = (float)(word >> 24) - 128.0f;
#pragma unroll
        for (int t = 0; t < MT; ++t) {
          // ring channel i of the row = source channel 4 w - sh + i = value 4 - sh + i of the two slices
          const float* v = a[u][t];
          const float av = sh == 0 ? v[4 + i] : (sh == 1 ? v[3 + i] : (sh == 2 ? v[2 + i] : v[1 + i]));
          asum[t] += av;
          acc[t][0] = fmaf(av, u0, acc[t][0]);
          acc[t][1] = fmaf(av, u1, acc[t][1]);
          acc[t][2] = fmaf(av, u2, acc[t][2]);
          acc[t][3] = fmaf(av, u3, acc[t][3]);
        }
      }
    }
  }
  // rows of the work-group through LDS, in their order
#pragma unroll
  for (int t = 0; t < MT; ++t) {
#pragma unroll
    for (int c = 0; c < 4; ++c) red[rsub][s_lane][t * 5 + c] = acc[t][c];
    red[rsub][s_lane][t * 5 + 4] = asum[t];
  }
  __syncthreads();
  if (rsub != 0) return;
  const size_t width = (size_t)p.ns * 4 + 4;
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    if (t >= p.m) break;
    float* out = p.partial + (((size_t)blockIdx.x * p.rows + row) * 4 + t) * width;
    float v[5] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int q = 0; q < RW; ++q) {
#pragma unroll
      for (int c = 0; c < 5; ++c) v[c] += red[q][s_lane][t * 5 + c];
    }
    if (slice_ok) *reinterpret_cast<float4*>(out + (size_t)ds * 4) = make_float4(v[0], v[1], v[2], v[3]);
    if (blockIdx.y == 0 && s_lane == 0) out[(size_t)p.ns * 4] = v[4];
  }
}

// Work-group = 16 output channels x 16 part lanes of one (dst row, token): lane q adds the parts
// q, q + 16, ... in their order, eight loads in flight at a time; the 16 lanes' sums are added in
// lane order, then the write-out.
template <typename T, typename DstT>
__global__ __launch_bounds__(256) void fc_w8_ring_finish_kernel(RingParams p) {
  __shared__ float red[16][16][2];
  const int n_all = p.ns * 4;
  const int cl = threadIdx.x & 15, q = threadIdx.x >> 4;
  const int n = blockIdx.x * 16 + cl;  // (n_all is a multiple of 4; the grid covers it in chunks of 16)
  const int t = blockIdx.y, row = blockIdx.z;
  const size_t width = (size_t)n_all + 4;
  const int nc = min(n, n_all - 1);
  float sum = 0.0f, asum = 0.0f;
  for (int part0 = q; part0 < p.parts; part0 += 16 * 8) {
    float v[8], av[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int part = min(part0 + 16 * j, p.parts - 1);
      const float* in = p.partial + (((size_t)part * p.rows + row) * 4 + t) * width;
      v[j] = in[nc];
      av[j] = in[n_all];
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (part0 + 16 * j < p.parts) {
        sum += v[j];
        asum += av[j];
      }
    }
  }
  red[q][cl][0] = sum;
  red[q][cl][1] = asum;
  __syncthreads();
  if (q != 0 || n >= n_all || (n >> 2) >= RingDstEndSlice(p)) return;
  sum = asum = 0.0f;
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    sum += red[j][cl][0];
    asum += red[j][cl][1];
  }
  int wb = p.batch_ids ? p.batch_ids[row] : 0;
  wb = min(max(wb, 0), p.weights_batch - 1);
  float s = p.scalar_scale, z = p.has_zero_point ? p.scalar_zero_point : 0.0f;
  if (p.scale_kind == kScaleLinear) {
    s = LoadF(static_cast<const T*>(p.scale), (size_t)wb * n_all + n);
    if (p.zero_point) z = LoadF(static_cast<const T*>(p.zero_point), (size_t)wb * n_all + n);
  }
  float r = s * fmaf(-z, asum, sum);
  if (RingSumInfinite(asum)) r = s * RingSumByProducts<T, false>(row, t, n, z);
  const size_t o = ((size_t)(n >> 2) * p.rows * p.m + (size_t)row * p.m + t) * 4 + (n & 3);
  DstT* dst = static_cast<DstT*>(p.dst);
  const DstT* bias = static_cast<const DstT*>(p.bias);
  if constexpr (std::is_same<DstT, float>::value) {
    dst[o] = bias ? r + bias[n] : r;
  } else {
    __half h = __float2half_rn(r);
    if (bias) h = __hadd(h, bias[n]);
    dst[o] = h;
  }
}

// ------------------------------------------------------------------------------------------
// The same walk in one launch: a work-group owns one output slice (4 channels) and MT tokens and walks
// the whole window by itself, so there are no partial sums and no second kernel.
//
// What bounds it: the dependent launch (1.55 us), then how fast a CU takes pieces that lie in lines of their
// own: a wave's load of 16-byte blocks a whole row (Ns x 16 bytes) apart touches 64 lines, its load of the
// activations of two tokens 32.  So the slice below a row's own comes from the neighbouring lane instead
// of memory and two tokens travel in one load (8 tokens x 8192 positions x 256 channels, a ring longer than that: 6.4 -> 5.8 us on
// one box, 6.6 on the box of the turn kernels' figures below; 74.7 us on the unspecialised kernel that served more than 4 tokens; one
// token 10.4 us with the window split, 5.0 here).  Neighbouring slices share the lines of the weights, so runs of 8 slices are
// dealt to one XCD, whose L2 fetches a line once.  A thread owns window rows tid, tid + THREADS, ...; the
// loads of two rows are in flight per thread, at 1024 threads a cache of 8192 positions at once.
// ------------------------------------------------------------------------------------------
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ half2_t AsHalf2(uint32_t v) { return __builtin_bit_cast(half2_t, v); }

// Sum over the 64 lanes of four values (lane l ends with value 2 * (l / 32) + (l / 16) % 2) by register
// exchanges that halve what a lane carries, then data-parallel moves over the 16 lanes that are left.
__device__ __forceinline__ float AddRow16(float v) {
  v += __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(v), 0x128 /* row_ror:8 */, 0xf, 0xf, false));
  const uint32_t up = __builtin_amdgcn_update_dpp(0u, __float_as_uint(v), 0x104 /* row_shl:4 */, 0xf, 0x5, false);
  const uint32_t both = __builtin_amdgcn_update_dpp(up, __float_as_uint(v), 0x114 /* row_shr:4 */, 0xf, 0xA, false);
  v += __uint_as_float(both);
  v += __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(v), 0x4E /* quad_perm:[2,3,0,1] */, 0xf, 0xf, false));
  v += __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(v), 0xB1 /* quad_perm:[1,0,3,2] */, 0xf, 0xf, false));
  return v;
}
__device__ __forceinline__ float SwapAdd32(float a, float b) {
  const u32x2 e = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(e[0]) + __uint_as_float(e[1]);
}
__device__ __forceinline__ float SwapAdd16(float a, float b) {
  const u32x2 e = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(e[0]) + __uint_as_float(e[1]);
}

// One slice of MT neighbouring tokens as it lies in memory: MT x 4 values in 32-bit words.
typedef uint32_t u32x4_word __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32x2_word __attribute__((ext_vector_type(2), aligned(4)));
template <typename T> constexpr int kWordsPerToken = (int)sizeof(T);
template <typename T, int MT>
__device__ __forceinline__ void LoadTokens(const T* p, size_t i, uint32_t (&v)[MT * kWordsPerToken<T>]) {
  if constexpr (MT * kWordsPerToken<T> == 2) {
    const u32x2_word r = *reinterpret_cast<const u32x2_word*>(p + i);
    v[0] = r[0];
    v[1] = r[1];
  } else {
#pragma unroll
    for (int q = 0; q < MT * kWordsPerToken<T> / 4; ++q) {
      const u32x4_word r = reinterpret_cast<const u32x4_word*>(p + i)[q];
#pragma unroll
      for (int j = 0; j < 4; ++j) v[q * 4 + j] = r[j];
    }
  }
}

// acc[c] += sum_i a_i (u_ic - 128) over one block (word i = ring channel i, byte c = output channel c) and
// asum += sum_i a_i, where a_i is value 4 - sh + i of the eight values {lo, hi}.
__device__ __forceinline__ void MultiplyRow(const float (&u)[4][4], const uint32_t* lo, const uint32_t* hi, int sh, float (&acc)[4],
                                            float& asum) {
  float v[8];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    v[i] = __uint_as_float(lo[i]);
    v[4 + i] = __uint_as_float(hi[i]);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float a = sh == 0 ? v[4 + i] : (sh == 1 ? v[3 + i] : (sh == 2 ? v[2 + i] : v[1 + i]));
    asum += a;
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[c] = fmaf(a, u[i][c], acc[c]);
  }
}
__device__ __forceinline__ void MultiplyRow(const half2_t (&u)[2][4], const uint32_t* lo, const uint32_t* hi, int sh, float (&acc)[4],
                                            float& asum) {
  // the words {y0, y1, y2} that hold halfs 4 - sh .. 7 - sh, shifted by one half where sh is odd
  const uint32_t y0 = sh == 0 ? hi[0] : (sh <= 2 ? lo[1] : lo[0]);
  const uint32_t y1 = sh == 0 ? hi[1] : (sh <= 2 ? hi[0] : lo[1]);
  const uint32_t y2 = sh <= 2 ? hi[1] : hi[0];
  const uint32_t by = (sh & 1) * 16;
  const half2_t a01 = AsHalf2(__builtin_amdgcn_alignbit(y1, y0, by)), a23 = AsHalf2(__builtin_amdgcn_alignbit(y2, y1, by));
  const half2_t one = {(_Float16)1.0f, (_Float16)1.0f};
  asum = __builtin_amdgcn_fdot2(a23, one, __builtin_amdgcn_fdot2(a01, one, asum, false), false);
#pragma unroll
  for (int c = 0; c < 4; ++c)
    acc[c] = __builtin_amdgcn_fdot2(a23, u[1][c], __builtin_amdgcn_fdot2(a01, u[0][c], acc[c], false), false);
}
// u - 128 of one block, in the form the multiply takes (fp16 tensors: pairs of input channels; exact)
__device__ __forceinline__ void Centre(const u32x4& blk, float (&u)[4][4]) {
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int c = 0; c < 4; ++c) u[i][c] = (float)((blk[i] >> (8 * c)) & 0xFFu) - 128.0f;
}
__device__ __forceinline__ void Centre(const u32x4& blk, half2_t (&u)[2][4]) {
  const half2_t off = {(_Float16)-1152.0f, (_Float16)-1152.0f};
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const uint32_t sel = 0x0c000c00u | (uint32_t)c | ((uint32_t)(4 + c) << 16);
      u[j][c] = AsHalf2(__builtin_amdgcn_perm(blk[2 * j + 1], blk[2 * j], sel) | 0x64006400u) + off;
    }
}
template <typename T> struct RingTypes;
template <> struct RingTypes<float> { typedef float centred[4][4]; };
template <> struct RingTypes<__half> { typedef half2_t centred[2][4]; };

// One result in the destination type, plus the bias
template <typename T>
__device__ __forceinline__ void RingStore(const RingParams& p, int n, size_t o, float r) {
  T* dst = static_cast<T*>(p.dst);
  const T* bias = static_cast<const T*>(p.bias);
  if constexpr (std::is_same<T, float>::value) {
    dst[o] = bias ? r + bias[n] : r;
  } else {
    __half h = __float2half_rn(r);
    if (bias) h = __hadd(h, bias[n]);
    dst[o] = h;
  }
}
// scale * (sum - zp * sum(a)) of output channel n (the rare second store comes last, out of the way of the first)
template <typename T, bool RING_O>
__device__ __forceinline__ void RingWrite(const RingParams& p, int wb, int n, size_t o, float sum, float asum, int row, int token) {
  float s = p.scalar_scale, z = p.has_zero_point ? p.scalar_zero_point : 0.0f;
  if (p.scale_kind == kScaleLinear) {
    s = LoadF(static_cast<const T*>(p.scale), (size_t)wb * p.ns * 4 + n);
    if (p.zero_point) z = LoadF(static_cast<const T*>(p.zero_point), (size_t)wb * p.ns * 4 + n);
  }
  RingStore<T>(p, n, o, s * fmaf(-z, asum, sum));
  if (RingSumInfinite(asum)) RingStore<T>(p, n, o, s * RingSumByProducts<T, RING_O>(row, token, n, z));
}

// (MT <= p.m: the last work-group along the tokens starts at token m - MT, and only it writes what is left)
template <typename T, int MT, int THREADS>
__global__ __launch_bounds__(THREADS) void fc_w8_ring_i_column_kernel(RingParams p) {
  constexpr int U = 2, WAVES = THREADS / 64, NW = kWordsPerToken<T>;
  __shared__ float red[WAVES][MT][5];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // runs of 8 slices on one XCD (work-groups go round-robin to the 8 of them); fewer than 8 runs: what one
  // of them does not hold at a time goes to others (20 channels, 16 rows of 49 tokens: all on XCD 0 else); not less, since
  // the tokens of a row share its weights, and the rows the lines of the activations
  constexpr int kSpreadShift = THREADS == 1024 ? 3 : 5;  // (8 slices x 8 or 32 token tiles fill 32 CUs)
  const int plane = blockIdx.z * ((p.m + MT - 1) / MT) + blockIdx.y;
  const int j = blockIdx.x >> 3, run = (blockIdx.x - ((plane >> kSpreadShift) & p.xcd_mask) * p.xcd_runs) & 7;
  const int ds = (j >> 3) * 64 + run * 8 + (j & 7);
  if (ds >= RingDstEndSlice(p)) return;  // (the whole work-group)
  const int row = blockIdx.z, tok_first = blockIdx.y * MT, tok0 = min(tok_first, p.m - MT);
  int wb = p.batch_ids ? p.batch_ids[row] : 0;
  wb = min(max(wb, 0), p.weights_batch - 1);
  const size_t act_stride = (size_t)p.src_rows * p.m;
  const T* act = static_cast<const T*>(p.act) + ((size_t)min(row, p.src_rows - 1) * p.m + tok0) * 4;
  const int off = ((p.params[p.ring_index] % p.ring_size) + p.ring_size) % p.ring_size;
  const int sh = off & 3, row0 = off >> 2;
  const int ks_end = RingSrcEndSlices(p);
  const int nrows = ks_end > 0 ? (sh + ks_end * 4 + 3) >> 2 : 0;  // window rows touched (at most ring_rows + 1)
  const u32x4* wcol = p.weights + (size_t)wb * p.ring_rows * p.ns + ds;

  float acc[MT][4], asum[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    asum[t] = 0.0f;
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[t][c] = 0.0f;
  }
  for (int base = wave * 64; base < nrows; base += THREADS * U) {  // (the same for the whole wave: lanes exchange below)
    u32x4 blk[U];
    uint32_t first[U][MT * NW], hi[U][MT * NW];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int w_wave = base + u * THREADS, w = w_wave + lane;
      int kb = row0 + min(w, nrows - 1);
      if (kb >= p.ring_rows) kb -= p.ring_rows;
      blk[u] = wcol[(size_t)kb * p.ns];
      // slice w holds source channels 4 w .. 4 w + 3; the row needs 4 w - sh .. 4 w - sh + 3, the rest of which is
      // the slice of the lane below (lane 0: a load of its own, one line for the wave)
      LoadTokens<T, MT>(act, (size_t)min(w, ks_end - 1) * act_stride * 4, hi[u]);
      LoadTokens<T, MT>(act, (size_t)max(min(w_wave, ks_end) - 1, 0) * act_stride * 4, first[u]);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int w = base + u * THREADS + lane;
      const bool lo_ok = w >= 1 && w - 1 < ks_end, hi_ok = w < ks_end;  // (a row past the window has neither)
      typename RingTypes<T>::centred cu;
      Centre(blk[u], cu);
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        uint32_t lo[NW], hv[NW];
#pragma unroll
        for (int i = 0; i < NW; ++i) {
          const uint32_t below = __builtin_amdgcn_update_dpp(first[u][t * NW + i], hi[u][t * NW + i], 0x138 /* wave_shr:1 */, 0xf, 0xf, false);
          lo[i] = lo_ok ? below : 0u;
          hv[i] = hi_ok ? hi[u][t * NW + i] : 0u;
        }
        MultiplyRow(cu, lo, hv, sh, acc[t], asum[t]);
      }
    }
  }
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const float v = AddRow16(SwapAdd16(SwapAdd32(acc[t][0], acc[t][2]), SwapAdd32(acc[t][1], acc[t][3])));
    const float s32 = SwapAdd32(asum[t], asum[t]);
    const float a = AddRow16(SwapAdd16(s32, s32));
    if ((lane & 15) == 0) red[wave][t][2 * (lane >> 5) + ((lane >> 4) & 1)] = v;
    if (lane == 0) red[wave][t][4] = a;
  }
  __syncthreads();
  if (tid >= MT * 4) return;
  const int t = tid >> 2, c = tid & 3;
  if (tok0 + t < tok_first) return;
  float sum = 0.0f, as = 0.0f;
#pragma unroll
  for (int q = 0; q < WAVES; ++q) {
    sum += red[q][t][c];
    as += red[q][t][4];
  }
  RingWrite<T, false>(p, wb, ds * 4 + c, ((size_t)ds * p.rows * p.m + (size_t)row * p.m + tok0 + t) * 4 + c, sum, as, row, tok0 + t);
}

// The same where the window is the whole ring and no runtime bound cuts it.  Then which rows are read does not depend on
// where the ring starts, only which source slices meet them: row r holds source channels 4 w - sh .. 4 w - sh + 3 with w = r - row0
// around the ring, whose first part is the slice of row r - 1, around the ring too.  So a thread walks the rows as they lie and
// requests its weights before the start of the ring is known, and scale and bias with the activations.  Each of the four shifts has a
// walk of its own, without selects, and without a zero point the sum of the activations is not needed.  8 tokens x 8192 positions x
// 256 channels 6.0 us (profiler figures; 6.6 in the column kernel; all activations through LDS, so that nothing but the reads
// from there waits for the start: 7.2).  One jump for the window and not one for every row and token: those were fetches of instructions
// that nothing had asked for, and took the kernel behind the column kernel where the activations are summed as well or
// a thread walks more than two rows (fp16, 367 random launches, geometric means of the speed over the column kernel's with a jump per
// row / one: no zero points, up to 2044 positions 1.06 / 1.10, up to 8192 1.08 / 1.10, more 1.02 / 1.06; zero points 0.99 / 1.04, 1.00 / 1.02,
// 0.96 / 1.01; fp32 1.11 .. 1.22 / 1.16 .. 1.27 and 1.10 .. 1.17 / 1.15 .. 1.23).
template <int SH>
__device__ __forceinline__ void MultiplyShifted(const float (&u)[4][4], const uint32_t* lo, const uint32_t* hi, bool zp, float (&acc)[4],
                                                float& asum) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float a = __uint_as_float(i < SH ? lo[4 - SH + i] : hi[i - SH]);
    if (zp) asum += a;
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[c] = fmaf(a, u[i][c], acc[c]);
  }
}
template <int SH>
__device__ __forceinline__ void MultiplyShifted(const half2_t (&u)[2][4], const uint32_t* lo, const uint32_t* hi, bool zp, float (&acc)[4],
                                                float& asum) {
  uint32_t a01, a23;
  if (SH == 0) {
    a01 = hi[0], a23 = hi[1];
  } else if (SH == 1) {
    a01 = __builtin_amdgcn_alignbit(hi[0], lo[1], 16), a23 = __builtin_amdgcn_alignbit(hi[1], hi[0], 16);
  } else if (SH == 2) {
    a01 = lo[1], a23 = hi[0];
  } else {
    a01 = __builtin_amdgcn_alignbit(lo[1], lo[0], 16), a23 = __builtin_amdgcn_alignbit(hi[0], lo[1], 16);
  }
  const half2_t one = {(_Float16)1.0f, (_Float16)1.0f};
  if (zp) asum = __builtin_amdgcn_fdot2(AsHalf2(a23), one, __builtin_amdgcn_fdot2(AsHalf2(a01), one, asum, false), false);
#pragma unroll
  for (int c = 0; c < 4; ++c)
    acc[c] = __builtin_amdgcn_fdot2(AsHalf2(a23), u[1][c], __builtin_amdgcn_fdot2(AsHalf2(a01), u[0][c], acc[c], false), false);
}
// Scale, zero point and bias of one output channel, requested ahead of their use
template <typename T>
struct RingChannel {
  float s, z;
  T bias;
};
template <typename T>
__device__ __forceinline__ RingChannel<T> LoadRingChannel(const RingParams& p, int wb, int n) {
  RingChannel<T> c = {p.scalar_scale, p.has_zero_point ? p.scalar_zero_point : 0.0f, T()};
  if (p.scale_kind == kScaleLinear) {
    c.s = LoadF(static_cast<const T*>(p.scale), (size_t)wb * p.ns * 4 + n);
    if (p.zero_point) c.z = LoadF(static_cast<const T*>(p.zero_point), (size_t)wb * p.ns * 4 + n);
  }
  if (p.bias) c.bias = static_cast<const T*>(p.bias)[n];
  return c;
}
template <typename T>
__device__ __forceinline__ void RingStoreChannel(const RingParams& p, const RingChannel<T>& c, size_t o, float r) {
  T* dst = static_cast<T*>(p.dst);
  if constexpr (std::is_same<T, float>::value) {
    dst[o] = p.bias ? r + c.bias : r;
  } else {
    __half h = __float2half_rn(r);
    if (p.bias) h = __hadd(h, c.bias);
    dst[o] = h;
  }
}

// The same of fp16 tensors as it lies in memory, hidden from the compiler until it is used: it moves the conversion of RingChannel up to the
// loads, and there the wave waits for them and for all loads before them.  (600 launches each of 16 .. 1024 x 256 .. 16384 channels, 1 .. 64
// tokens, without that wait: values 1.01 times as fast in the geometric mean, keys without zero points 1.01; keys with zero points, whose end
// takes longer then, 0.99.)
struct RingChannelRaw {
  uint32_t s, z, bias;
};
__device__ __forceinline__ RingChannelRaw LoadRingChannelRaw(const RingParams& p, int wb, int n) {
  RingChannelRaw c = {0u, 0u, 0u};
  const size_t at = (size_t)wb * p.ns * 4 + n;
  if (p.scale_kind == kScaleLinear) c.s = static_cast<const uint16_t*>(p.scale)[at];
  if (p.scale_kind == kScaleLinear && p.zero_point) c.z = static_cast<const uint16_t*>(p.zero_point)[at];
  if (p.bias) c.bias = static_cast<const uint16_t*>(p.bias)[n];
  return c;
}
__device__ __forceinline__ __half RingChannelValue(uint32_t raw) {
  asm volatile("" : "+v"(raw));
  return __ushort_as_half((unsigned short)raw);
}
// scale * (sum - zp * asum) plus the bias (the rare second store comes last, out of the way of the first)
template <bool RING_O, bool ZP>
__device__ __forceinline__ void RingStoreChannelRaw(const RingParams& p, const RingChannelRaw& c, int n, size_t o, float sum, float asum, int row,
                                                    int token) {
  float s = p.scalar_scale, z = p.scalar_zero_point;
  if (p.scale_kind == kScaleLinear) {
    s = __half2float(RingChannelValue(c.s));
    if (ZP && p.zero_point) z = __half2float(RingChannelValue(c.z));
  }
  const __half bias = RingChannelValue(c.bias);
  auto store = [&](float r) {
    __half h = __float2half_rn(r);
    if (p.bias) h = __hadd(h, bias);
    static_cast<__half*>(p.dst)[o] = h;
  };
  store(s * (ZP ? fmaf(-z, asum, sum) : sum));
  if (ZP && RingSumInfinite(asum)) store(s * RingSumByProducts<__half, RING_O>(row, token, n, z));
}

template <typename F>
__device__ __forceinline__ void WithShift(int sh, F f) {
  if (sh == 0) f(std::integral_constant<int, 0>());
  else if (sh == 1) f(std::integral_constant<int, 1>());
  else if (sh == 2) f(std::integral_constant<int, 2>());
  else f(std::integral_constant<int, 3>());
}
// Token slots with which the kernel below is there for launches with zero points (ColumnTurns)
template <typename T, int THREADS>
constexpr bool TurnWithZeroPoint(int slots) { return std::is_same<T, float>::value || THREADS == 256 || slots <= 2; }

// Token slots with which 1024 threads of the kernel below come in two forms: one work-group per CU (ALONE), two.  Where there is no more than one
// for every CU of an XCD, two of them are put on one CU all the same where they fit: fp32, 11 tokens x 7172 positions x 16 channels 6.2 us,
// alone 4.9.  Where there are more, two on a CU hide each other's waits (speed over the column kernel's, geometric means of random
// launches of 1.25 .. 2 per CU: two fp32 tokens 1.22, alone 1.07; four fp16 tokens 1.27 and 1.15).
template <typename T, int THREADS>
constexpr bool TurnAloneOrNot(int slots) { return THREADS == 1024 && sizeof(T) * slots == 8; }

// (MT as in the column kernel; work-groups are dealt to the XCDs as there)
template <typename T, int MT, int THREADS, bool ZP, bool ALONE = false>
__global__ __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(THREADS / 256, ALONE ? THREADS / 256 : 8))) void fc_w8_ring_i_turn_kernel(RingParams p) {
  constexpr int U = 2, WAVES = THREADS / 64, NW = kWordsPerToken<T>;
  constexpr bool RAW = std::is_same<T, __half>::value;  // (RingChannelRaw)
  __shared__ float red[WAVES][MT][5];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  constexpr int kSpreadShift = THREADS == 1024 ? 3 : 5;
  const int plane = blockIdx.z * ((p.m + MT - 1) / MT) + blockIdx.y;
  const int j = blockIdx.x >> 3, run = (blockIdx.x - ((plane >> kSpreadShift) & p.xcd_mask) * p.xcd_runs) & 7;
  const int ds = (j >> 3) * 64 + run * 8 + (j & 7);
  if (ds >= p.ns) return;  // (the whole work-group)
  const int row = blockIdx.z, tok_first = blockIdx.y * MT, tok0 = min(tok_first, p.m - MT);
  int wb = p.batch_ids ? p.batch_ids[row] : 0;
  wb = min(max(wb, 0), p.weights_batch - 1);
  const int rows = p.ring_rows;
  const u32x4* wcol = p.weights + (size_t)wb * rows * p.ns + ds;
  const size_t act_stride = (size_t)p.src_rows * p.m * 4;
  const T* act = static_cast<const T*>(p.act) + ((size_t)min(row, p.src_rows - 1) * p.m + tok0) * 4;
  u32x4 blk[U];
  auto load_row = [&](int first_row) { return wcol[(size_t)min(first_row + lane, rows - 1) * p.ns]; };
#pragma unroll
  for (int u = 0; u < U; ++u) blk[u] = load_row(wave * 64 + u * THREADS);
  __builtin_amdgcn_sched_barrier(0);
  const int off = ((p.params[p.ring_index] % p.ring_size) + p.ring_size) % p.ring_size;
  const int sh = off & 3, row0 = off >> 2;
  std::conditional_t<RAW, RingChannelRaw, RingChannel<T>> channel;
  if (tid < MT * 4) {
    if constexpr (RAW) channel = LoadRingChannelRaw(p, wb, ds * 4 + (tid & 3));
    else channel = LoadRingChannel<T>(p, wb, ds * 4 + (tid & 3));
  }

  float acc[MT][4], asum[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    asum[t] = 0.0f;
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[t][c] = 0.0f;
  }
  // The window, with SH (0 .. 3) for the ring's start against a slice or, where SH is 4, with sh looked at for every row and token
  auto walk = [&](auto shift) {
    constexpr int SH = decltype(shift)::value;
    for (int base = wave * 64; base < rows; base += THREADS * U) {  // (the same for the whole wave: lanes exchange below)
      uint32_t first[U][MT * NW], hi[U][MT * NW];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int r0 = min(base + u * THREADS, rows - 1);  // (the wave's first row)
        const int below = r0 - row0 + (r0 > row0 ? -1 : rows - 1);
        int w = min(r0 + lane, rows - 1) - row0;
        w = w < 0 ? w + rows : w;
        LoadTokens<T, MT>(act, (size_t)w * act_stride, hi[u]);
        LoadTokens<T, MT>(act, (size_t)below * act_stride, first[u]);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const bool live = base + u * THREADS + lane < rows;  // (rows past the ring's last one count as zero)
        typename RingTypes<T>::centred cu;
        Centre(blk[u], cu);
#pragma unroll
        for (int t = 0; t < MT; ++t) {
          auto multiply = [&](auto row_shift) {
            constexpr int S = decltype(row_shift)::value;
            uint32_t lo[NW], hv[NW];
#pragma unroll
            for (int i = 0; i < NW; ++i) {
              if (S > 0) {
                lo[i] = __builtin_amdgcn_update_dpp(first[u][t * NW + i], hi[u][t * NW + i], 0x138 /* wave_shr:1 */, 0xf, 0xf, false);
                lo[i] = live ? lo[i] : 0u;
              }
              hv[i] = live ? hi[u][t * NW + i] : 0u;
            }
            MultiplyShifted<S>(cu, lo, hv, ZP, acc[t], asum[t]);
          };
          if constexpr (SH < 4) multiply(shift);
          else WithShift(sh, multiply);
        }
        if (base + THREADS * U < rows) blk[u] = load_row(base + THREADS * U + u * THREADS);
      }
    }
  };
  // (four fp16 tokens: four walks are 73 registers, one work-group of 1024 threads per CU; with a jump for every row and token 61)
  if constexpr (std::is_same<T, __half>::value && TurnAloneOrNot<T, THREADS>(MT) && !ALONE) walk(std::integral_constant<int, 4>());
  else WithShift(sh, walk);
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const float v = AddRow16(SwapAdd16(SwapAdd32(acc[t][0], acc[t][2]), SwapAdd32(acc[t][1], acc[t][3])));
    if ((lane & 15) == 0) red[wave][t][2 * (lane >> 5) + ((lane >> 4) & 1)] = v;
    if (ZP) {
      const float s32 = SwapAdd32(asum[t], asum[t]);
      const float a = AddRow16(SwapAdd16(s32, s32));
      if (lane == 0) red[wave][t][4] = a;
    }
  }
  __syncthreads();
  if (tid >= MT * 4) return;
  const int t = tid >> 2, c = tid & 3, n = ds * 4 + c;
  if (tok0 + t < tok_first) return;
  float sum = 0.0f, as = 0.0f;
#pragma unroll
  for (int q = 0; q < WAVES; ++q) {
    sum += red[q][t][c];
    if (ZP) as += red[q][t][4];
  }
  const size_t o = ((size_t)ds * p.rows * p.m + (size_t)row * p.m + tok0 + t) * 4 + c;
  if constexpr (RAW) {
    RingStoreChannelRaw<false, ZP>(p, channel, n, o, sum, as, row, tok0 + t);
  } else {
    RingStoreChannel<T>(p, channel, o, channel.s * (ZP ? fmaf(-channel.z, as, sum) : sum));
    if (ZP && RingSumInfinite(as)) RingStore<T>(p, n, o, channel.s * RingSumByProducts<T, false>(row, tok0 + t, n, channel.z));
  }
}

// ------------------------------------------------------------------------------------------
// Ring over the output channels of a kOSpatialIOGroupO4I4 buffer (GetRingedOAddresses,
// fully_connected.cc:411-422, 680-697): query x key cache.  Word (ks, o) of the buffer holds input
// channels 4 ks .. 4 ks + 3 of ring channel o, one per byte; dst channel c is ring channel
// (c + offset) % ring_size.  A thread owns one dst slice, whose four words lie one after the other
// (one 16-byte load from a 4-byte boundary), except in the slice that the end of the ring cuts.
//
// Work-group = 16 slices x 16 K lanes (K-slices k, k + 16, ...; 4 of them in a wave), MT tokens.  What bounds
// it is latency: the ring's start has to be read before the first weight address is known.  So the
// activations, which do not depend on it, go to LDS meanwhile (the 16 lanes of a K-slice read the same
// 8 or 16 bytes per token), the weights of four K-slices per thread are then in flight at once, and the
// sums meet by register exchanges inside a wave and through 4 KB of LDS across the waves.  8 tokens x 8192
// positions x 256 channels of a longer ring, 2.1 MB: 4.0 us (5.3 with the activations from memory and the whole reduction
// through LDS, 10.1 us on the unspecialised kernel that served it; 4.5 on the box of the turn kernels' figures below).
// ------------------------------------------------------------------------------------------
__device__ __forceinline__ void CentreO(const u32x4& w, float (&u)[4][4]) {
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int c = 0; c < 4; ++c) u[i][c] = (float)((w[c] >> (8 * i)) & 0xFFu) - 128.0f;
}
__device__ __forceinline__ void CentreO(const u32x4& w, half2_t (&u)[2][4]) {
  const half2_t off = {(_Float16)-1152.0f, (_Float16)-1152.0f};
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    u[0][c] = AsHalf2(__builtin_amdgcn_perm(0u, w[c], 0x0c010c00u) | 0x64006400u) + off;
    u[1][c] = AsHalf2(__builtin_amdgcn_perm(0u, w[c], 0x0c030c02u) | 0x64006400u) + off;
  }
}

template <typename T, int MT>
__global__ __launch_bounds__(256) void fc_w8_ring_o_kernel(RingParams p) {
  constexpr int KL = 16, U = 4, NW = kWordsPerToken<T>, CHUNK = 256;  // K-slices staged at a time
  __shared__ uint32_t acts[CHUNK][MT * NW];
  __shared__ float red[4][MT][64], reda[4][MT];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, sl = tid & 15, kl = tid >> 4;
  const int row = blockIdx.z, tok_first = blockIdx.y * MT, tok0 = min(tok_first, p.m - MT);
  const size_t act_stride = (size_t)p.src_rows * p.m;
  const T* act = static_cast<const T*>(p.act) + ((size_t)min(row, p.src_rows - 1) * p.m + tok0) * 4;
  const int ks_end = RingSrcEndSlices(p), ns_end = RingDstEndSlice(p);
  if ((int)blockIdx.x * 16 >= ns_end) return;  // (the whole work-group)
  const int ds = min((int)blockIdx.x * 16 + sl, p.ns - 1);
  int wb = p.batch_ids ? p.batch_ids[row] : 0;
  wb = min(max(wb, 0), p.weights_batch - 1);
  const int off = ((p.params[p.ring_index] % p.ring_size) + p.ring_size) % p.ring_size;
  const uint32_t* w32 = reinterpret_cast<const uint32_t*>(p.weights) + (size_t)wb * p.ks * p.ring_size;
  const int o0 = (int)(((long)ds * 4 + off) % p.ring_size);
  const bool whole = o0 + 4 <= p.ring_size;
  float acc[MT][4], asum[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    asum[t] = 0.0f;
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[t][c] = 0.0f;
  }
  for (int chunk = 0; chunk < ks_end; chunk += CHUNK) {
    const int count = min(ks_end - chunk, CHUNK);
    if (chunk > 0) __syncthreads();  // (everybody is done with the chunk before)
    for (int i = tid; i < count; i += 256) {
      uint32_t v[MT * NW];
      LoadTokens<T, MT>(act, (size_t)(chunk + i) * act_stride * 4, v);
#pragma unroll
      for (int q = 0; q < MT * NW; ++q) acts[i][q] = v[q];
    }
    bool staged = false;
    for (int k0 = kl; k0 < count || !staged; k0 += KL * U) {
      u32x4 w[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const uint32_t* base = w32 + (size_t)(chunk + min(k0 + u * KL, count - 1)) * p.ring_size;
        if (whole) {
          w[u] = *reinterpret_cast<const u32x4_word*>(base + o0);
        } else {
#pragma unroll
          for (int c = 0; c < 4; ++c) w[u][c] = base[o0 + c < p.ring_size ? o0 + c : o0 + c - p.ring_size];
        }
      }
      if (!staged) __syncthreads();  // (once per chunk and thread: the first pass of every thread)
      staged = true;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k = k0 + u * KL;
        if (k < count) {
          typename RingTypes<T>::centred cu;
          CentreO(w[u], cu);
          uint32_t v[MT * NW];
#pragma unroll
          for (int q = 0; q < MT * NW; ++q) v[q] = acts[k][q];
#pragma unroll
          for (int t = 0; t < MT; ++t) MultiplyRow(cu, v + t * NW, v + t * NW, 0, acc[t], asum[t]);
        }
      }
    }
  }
  // lane = slice + 16 x K lane of the wave; two exchanges leave it with channel 2 * (lane / 32) + (lane / 16) % 2
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    red[wave][t][lane] = SwapAdd16(SwapAdd32(acc[t][0], acc[t][2]), SwapAdd32(acc[t][1], acc[t][3]));
    const float s32 = SwapAdd32(asum[t], asum[t]);
    const float a = SwapAdd16(s32, s32);
    if (lane == 0) reda[wave][t] = a;
  }
  __syncthreads();
  if (tid >= MT * 64) return;
  const int c = tid & 3, t = (tid >> 2) % MT, s = (tid >> 2) / MT;
  const int slice = blockIdx.x * 16 + s;
  if (slice >= ns_end || tok0 + t < tok_first) return;
  float sum = 0.0f, as = 0.0f;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    sum += red[q][t][c * 16 + s];
    as += reda[q][t];
  }
  RingWrite<T, true>(p, wb, slice * 4 + c, ((size_t)slice * p.rows * p.m + (size_t)row * p.m + tok0 + t) * 4 + c, sum, as, row, tok0 + t);
}

// The same where every channel of the ring is a dst channel: a work-group takes 64 channels as they lie in the ring, so no
// address of the weights or activations depends on where the ring starts, only the dst channels that the sums are for.
// 8 tokens x 8192 positions x 256 channels 4.5 -> 3.9 us (profiler figures; a step of 18 layers, keys and values, 189 -> 176 us when both kernels
// were new.  All kernel arguments in one batch of scalar loads at the top, in both: 12 us a step more).
template <typename T, int MT, bool ZP>
__global__ __launch_bounds__(256) void fc_w8_ring_o_turn_kernel(RingParams p) {
  constexpr int KL = 16, U = 4, NW = kWordsPerToken<T>, CHUNK = 256;
  constexpr bool RAW = std::is_same<T, __half>::value && !ZP;  // (RingChannelRaw)
  __shared__ uint32_t acts[CHUNK][MT * NW];
  __shared__ float red[4][MT][64], reda[4][MT];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, sl = tid & 15, kl = tid >> 4;
  const int row = blockIdx.z, tok_first = blockIdx.y * MT, tok0 = min(tok_first, p.m - MT);
  const size_t act_stride = (size_t)p.src_rows * p.m;
  const T* act = static_cast<const T*>(p.act) + ((size_t)min(row, p.src_rows - 1) * p.m + tok0) * 4;
  const int ks_end = RingSrcEndSlices(p);
  int wb = p.batch_ids ? p.batch_ids[row] : 0;
  wb = min(max(wb, 0), p.weights_batch - 1);
  const uint32_t* w32 = reinterpret_cast<const uint32_t*>(p.weights) + (size_t)wb * p.ks * p.ring_size + min((int)blockIdx.x * 16 + sl, p.ns - 1) * 4;
  float acc[MT][4], asum[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    asum[t] = 0.0f;
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[t][c] = 0.0f;
  }
  // the sum that this thread finishes: channel c of slice s of the ring for token t
  const int c = tid & 3, t_out = (tid >> 2) % MT, s = (tid >> 2) / MT;
  int n = 0;
  std::conditional_t<RAW, RingChannelRaw, RingChannel<T>> channel;
  for (int chunk = 0; chunk < ks_end || chunk == 0; chunk += CHUNK) {
    const int count = min(ks_end - chunk, CHUNK);
    if (chunk > 0) __syncthreads();  // (everybody is done with the chunk before)
    u32x4 w[U];
    auto load_weights = [&](int k0) {
#pragma unroll
      for (int u = 0; u < U; ++u)
        w[u] = *reinterpret_cast<const u32x4_word*>(w32 + (size_t)max(chunk + min(k0 + u * KL, count - 1), 0) * p.ring_size);
    };
    load_weights(kl);
    for (int i = tid; i < count; i += 256) {
      uint32_t v[MT * NW];
      LoadTokens<T, MT>(act, (size_t)(chunk + i) * act_stride * 4, v);
#pragma unroll
      for (int q = 0; q < MT * NW; ++q) acts[i][q] = v[q];
    }
    if (chunk == 0) {
      const int off = ((p.params[p.ring_index] % p.ring_size) + p.ring_size) % p.ring_size;
      n = (blockIdx.x * 16 + s) * 4 + c - off;
      n = n < 0 ? n + p.ring_size : n;
      if (tid < MT * 64 && (int)blockIdx.x * 16 + s < p.ns) {
        if constexpr (RAW) channel = LoadRingChannelRaw(p, wb, n);
        else channel = LoadRingChannel<T>(p, wb, n);
      }
    }
    __syncthreads();
    for (int k0 = kl; k0 < count; k0 += KL * U) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k = k0 + u * KL;
        if (k < count) {
          typename RingTypes<T>::centred cu;
          CentreO(w[u], cu);
          uint32_t v[MT * NW];
#pragma unroll
          for (int q = 0; q < MT * NW; ++q) v[q] = acts[k][q];
#pragma unroll
          for (int t = 0; t < MT; ++t) MultiplyShifted<0>(cu, v + t * NW, v + t * NW, ZP, acc[t], asum[t]);
        }
      }
      if (k0 + KL * U < count) load_weights(k0 + KL * U);
    }
  }
  // lane = slice + 16 x K lane of the wave; two exchanges leave it with channel 2 * (lane / 32) + (lane / 16) % 2
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    red[wave][t][lane] = SwapAdd16(SwapAdd32(acc[t][0], acc[t][2]), SwapAdd32(acc[t][1], acc[t][3]));
    if (ZP) {
      const float s32 = SwapAdd32(asum[t], asum[t]);
      const float a = SwapAdd16(s32, s32);
      if (lane == 0) reda[wave][t] = a;
    }
  }
  __syncthreads();
  if (tid >= MT * 64 || (int)blockIdx.x * 16 + s >= p.ns || tok0 + t_out < tok_first) return;
  float sum = 0.0f, as = 0.0f;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    sum += red[q][t_out][c * 16 + s];
    if (ZP) as += reda[q][t_out];
  }
  const size_t o = ((size_t)(n >> 2) * p.rows * p.m + (size_t)row * p.m + tok0 + t_out) * 4 + (n & 3);
  if constexpr (RAW) {
    RingStoreChannelRaw<true, ZP>(p, channel, n, o, sum, as, row, tok0 + t_out);
  } else {
    RingStoreChannel<T>(p, channel, o, channel.s * (ZP ? fmaf(-channel.z, as, sum) : sum));
    if (ZP && RingSumInfinite(as)) RingStore<T>(p, n, o, channel.s * RingSumByProducts<T, true>(row, tok0 + t_out, n, channel.z));
  }
}

// turn: 0: column kernel; 1: turn kernel; 2: turn kernel, one work-group per CU where there is a form for that
template <typename T, int MT, int THREADS>
hipError_t LaunchColumnT(const RingParams& p, int turn, hipStream_t stream) {
  const dim3 grid(DivUp(p.ns, 64) * 64, DivUp(p.m, MT), p.rows), block(THREADS);
  if (turn > 0 && !p.has_zero_point) {
    if (TurnAloneOrNot<T, THREADS>(MT) && turn == 2)
      hipLaunchKernelGGL((fc_w8_ring_i_turn_kernel<T, MT, THREADS, false, TurnAloneOrNot<T, THREADS>(MT)>), grid, block, 0, stream, p);
    else
      hipLaunchKernelGGL((fc_w8_ring_i_turn_kernel<T, MT, THREADS, false>), grid, block, 0, stream, p);
    return hipGetLastError();
  }
  if constexpr (TurnWithZeroPoint<T, THREADS>(MT)) {
    if (turn > 0) {
      hipLaunchKernelGGL((fc_w8_ring_i_turn_kernel<T, MT, THREADS, true>), grid, block, 0, stream, p);
      return hipGetLastError();
    }
  }
  hipLaunchKernelGGL((fc_w8_ring_i_column_kernel<T, MT, THREADS>), grid, block, 0, stream, p);
  return hipGetLastError();
}
template <typename T>
hipError_t LaunchColumn(const RingParams& p, int slots, bool small, int turn, hipStream_t stream) {
  if (slots == 4) return small ? LaunchColumnT<T, 4, 256>(p, turn, stream) : LaunchColumnT<T, 4, 1024>(p, turn, stream);
  if (slots == 2) return small ? LaunchColumnT<T, 2, 256>(p, turn, stream) : LaunchColumnT<T, 2, 1024>(p, turn, stream);
  return small ? LaunchColumnT<T, 1, 256>(p, turn, stream) : LaunchColumnT<T, 1, 1024>(p, turn, stream);
}
template <typename T, int MT>
hipError_t LaunchRingOT(const RingParams& p, bool turn, hipStream_t stream) {
  const dim3 grid(DivUp(p.ns, 16), DivUp(p.m, MT), p.rows), block(256);
  if (turn && p.has_zero_point)
    hipLaunchKernelGGL((fc_w8_ring_o_turn_kernel<T, MT, true>), grid, block, 0, stream, p);
  else if (turn)
    hipLaunchKernelGGL((fc_w8_ring_o_turn_kernel<T, MT, false>), grid, block, 0, stream, p);
  else
    hipLaunchKernelGGL((fc_w8_ring_o_kernel<T, MT>), grid, block, 0, stream, p);
  return hipGetLastError();
}
template <typename T>
hipError_t LaunchRingO(const RingParams& p, int slots, bool turn, hipStream_t stream) {
  if (slots == 4) return LaunchRingOT<T, 4>(p, turn, stream);
  if (slots == 2) return LaunchRingOT<T, 2>(p, turn, stream);
  return LaunchRingOT<T, 1>(p, turn, stream);
}

template <typename T, int LS>
hipError_t LaunchRingT(const RingParams& p, bool dst_f16, hipStream_t stream) {
  const dim3 grid(p.parts, DivUp(p.ns, LS), p.rows);
  if (p.m == 1)
    hipLaunchKernelGGL((fc_w8_ring_i_kernel<T, LS, 1>), grid, dim3(kRingThreads), 0, stream, p);
  else if (p.m == 2)
    hipLaunchKernelGGL((fc_w8_ring_i_kernel<T, LS, 2>), grid, dim3(kRingThreads), 0, stream, p);
  else
    hipLaunchKernelGGL((fc_w8_ring_i_kernel<T, LS, 4>), grid, dim3(kRingThreads), 0, stream, p);
  const dim3 fgrid(DivUp(p.ns * 4, 16), p.m, p.rows);
  if (dst_f16)
    hipLaunchKernelGGL((fc_w8_ring_finish_kernel<T, __half>), fgrid, dim3(256), 0, stream, p);
  else
    hipLaunchKernelGGL((fc_w8_ring_finish_kernel<T, float>), fgrid, dim3(256), 0, stream, p);
  return hipGetLastError();
}

}  // namespace

size_t FcW8RingWorkspaceFloats(int max_tokens, int o) {
  const int n_pad = DivUp(o, 4) * 4;
  // (a launch's dst rows x tokens per row are at most max_tokens; every row keeps 4 token slots)
  const size_t rows_tokens = (size_t)std::min(std::max(max_tokens, 1), 16) * 4;
  return std::min((size_t)kRingMaxParts * rows_tokens * (n_pad + 4), (size_t)8 << 20);
}

bool RingShapeOk(const FcArgs& a) {
  if (a.params == nullptr || a.weight_bits != 8 || a.ring_size < 4 || a.ring_size % 4 != 0) return false;
  if (a.packed_params_offset >= 0 || a.scale_kind == kScaleBlock || a.act_f16 != a.dst_f16) return false;
  // one output group (more dst channels than a ring over the output channels holds: refused by the unspecialised kernel)
  const int ns = DivUp(a.n, 4);
  if (EffectiveGroup(a.group, ns) != ns) return false;
  return a.m >= 1 && a.rows >= 1 && a.rows <= 65535;
}
bool PartsSupported(const FcArgs& a) {
  if (a.m > 4 || (long)a.rows * a.m > 16 || a.partial == nullptr) return false;
  // at least one part must fit the workspace
  return (size_t)a.rows * 4 * ((size_t)DivUp(a.n, 4) * 4 + 4) <= a.partial_floats;
}

int RingWindow(const FcArgs& a) { return std::min(DivUp(a.k, 4), a.ring_size / 4) + 1; }

// Token slots of a column work-group: two, so that the slices of a narrow cache (64 for a head of 256) occupy the chip
// (8 tokens x 8192 positions x 256 channels: 5.8 us, 8.6 with one slot, 6.2 with four); four where they do anyway
// (4096 positions x 512 channels: 5.25 against 5.8 us).
int ColumnSlots(const FcArgs& a) {
  int slots = (long)DivUp(a.n, 4) * a.rows * DivUp(a.m, 4) >= 256 ? 4 : 2;
  while (slots > a.m) slots /= 2;
  return slots;
}

// The split window: lanes along the output slices (a power of two up to 64) and parts of about 32 KB of weights each, at most
// what the workspace holds.
struct RingSplit {
  int lanes, parts, rows_in_flight;
};
RingSplit SplitWindow(const FcArgs& a) {
  const int ns = DivUp(a.n, 4), window = RingWindow(a);
  RingSplit r;
  r.lanes = 16;
  while (r.lanes < 64 && r.lanes < ns) r.lanes *= 2;
  r.rows_in_flight = kRingThreads / r.lanes * RingUnroll(a.m == 1 ? 1 : (a.m == 2 ? 2 : 4));
  const size_t bytes = (size_t)window * ns * 16;
  int parts = (int)std::min<size_t>(kRingMaxParts, std::max<size_t>(1, bytes / 32768));
  parts = std::min(parts, std::max(1, DivUp(window, r.rows_in_flight)));
  const size_t per_part = (size_t)a.rows * 4 * ((size_t)ns * 4 + 4);
  r.parts = std::max(1, (int)std::min<size_t>(parts, a.partial_floats / per_part));
  return r;
}

// Which kernel takes the ring over the input channels.  A column work-group reads 16 bytes of a line of its own per window row, so
// its time grows with window x slices x token tiles over the CUs (2000 positions x 2500 channels x 39 tokens 2150 us, the
// unspecialised kernel 560); the split window reads whole lines but is two launches with 32 activations per row and thread (8192
// positions x 256 channels, one token: 10.4 us, 5.0 in columns; 3088 x 2352, 16 rows of one token: 24 against 73).  Times in us, each
// the root of the sum of squares of a work-group's chain and of the busiest share of the work, plus the weights' bytes; fitted to
// 9319 random launches (windows of 128 .. 65536 positions, 4 .. 8192 channels, 1 .. 64 tokens x 1 .. 16 rows, fp16 and fp32) to
// within 17 % in nine of ten.  Their choice is slower than what served these launches without the column kernel by more than 10 %
// in 49 of them (in 1625 if it takes them all).
double RingMegabytes(const FcArgs& a) { return 16e-6 * a.rows * DivUp(a.n, 4) * RingWindow(a); }
// work-groups per CU of the busiest XCD, as the column and the turn kernel deal them
double ColumnGroupsPerCu(const FcArgs& a, int slots, bool small) {
  const int ns = DivUp(a.n, 4), runs = std::min(8, DivUp(ns, 8)), copies = runs == 1 ? 8 : (runs == 2 ? 4 : (runs <= 4 ? 2 : 1));
  const long planes = (long)DivUp(a.m, slots) * a.rows, together = small ? 32 : 8;
  const long shared = planes <= together ? planes : std::max(together, (planes + copies - 1) / copies);
  return (ns / 64 * 8 + std::min(8, ns % 64)) * (double)shared / 32.0;
}
double ColumnUs(const FcArgs& a) {
  struct Cost {
    double pass, row, act, group;  // per pass of 1024 threads; per 1000 rows: weights, activations; per work-group of 1024 threads
  };
  static const Cost kCost[2][3] = {{{1.5, 1.4, 0.82, 0.18}, {1.8, 1.2, 0.83, 0.46}, {4.3, 1.5, 0.68, 1.1}},   // fp16: 1, 2, 4 slots
                                   {{1.7, 1.2, 0.65, 0.49}, {2.6, 1.2, 0.72, 1.2}, {8.5, 2.0, 0.49, 2.9}}};  // fp32
  const int window = RingWindow(a), slots = ColumnSlots(a);
  const bool small = window <= 512;
  const Cost& c = kCost[a.act_f16 ? 0 : 1][slots == 1 ? 0 : (slots == 2 ? 1 : 2)];
  const double cus = ColumnGroupsPerCu(a, slots, small);
  const double lines = std::min(1.0, a.src_rows * (double)a.m * (a.act_f16 ? 8 : 16) / 128.0);  // lines that a row's activations touch
  const double chain = small ? 0.0 : std::max(1.0, std::ceil(cus / 2.0)) * DivUp(window, 2048) * c.pass;
  const double work = cus * (window * (c.row + c.act * lines) / 1000.0 + c.group * (small ? 0.31 : 1.0));
  return 3.0 + std::hypot(chain, work) + 0.16 * RingMegabytes(a);
}
double SplitUs(const FcArgs& a) {
  struct Cost {
    double fixed, pass, group, sum;
  };
  static const Cost kCost[3] = {{4.1, 2.7, 0.66, 1.5}, {5.0, 2.4, 0.88, 1.0}, {4.4, 4.7, 2.2, 1.7}};  // 1, 2, 3..4 tokens
  const RingSplit r = SplitWindow(a);
  const Cost& c = kCost[a.m == 1 ? 0 : (a.m == 2 ? 1 : 2)];
  const double groups = (double)r.parts * DivUp(DivUp(a.n, 4), r.lanes) * a.rows;
  const int passes = DivUp(DivUp(RingWindow(a), r.parts), r.rows_in_flight);
  return c.fixed + std::hypot(std::max(1.0, std::ceil(groups / 512)) * passes * c.pass, groups / 256 * c.group) +
         DivUp(r.parts, 128) * c.sum + 0.16 * DivUp(a.n, 4) * 4 * a.m * a.rows / 4096 + 0.055 * RingMegabytes(a);
}
double UnspecialisedUs(const FcArgs& a) {
  const double groups = (double)DivUp(DivUp(a.n, 4), 16) * DivUp(a.m, 4) * a.rows, steps = DivUp(a.k, 64);
  return 5.9 + std::hypot(0.74 * steps, groups / 256 * (0.47 * steps + 1.1)) + 0.24 * RingMegabytes(a);
}
// Whether the turn kernel takes a launch from the column kernel: the window is the whole ring and no runtime bound cuts it.  With zero points the
// activations are summed as in the column kernel, and what is left is the earlier start and the selects.  fp16 (random launches, speed over
// the column kernel's, geometric mean and least): a thread's two rows cover the ring 1.03, 0.93; more rows 1.01, 0.94; four slots of 1024 threads
// 1.00, 0.90: there it is ahead only where the ring starts on a whole slice.  fp32 1.05 .. 1.5, but with two slots 1024 threads are 67
// registers each, 58 in the column kernel: one work-group per CU instead of two; at 1.25 of them per CU still 1.05 .. 1.08, from 1.5 on 0.98, 0.87.
bool ColumnTurns(const FcArgs& a, int slots, bool small) {
  if (a.k != a.ring_size || a.src_end_ch_index >= 0 || a.dst_end_ch_index >= 0) return false;
  if (!a.has_zero_point) return true;
  if (a.act_f16)
    return (small ? TurnWithZeroPoint<__half, 256>(slots) : TurnWithZeroPoint<__half, 1024>(slots)) && a.ring_size / 4 <= (small ? 512 : 2048);
  return slots != 2 || small || ColumnGroupsPerCu(a, slots, small) <= 1.25;
}
// (longer windows were not measured in columns, but at 8192 rows x 256 channels and one token: 12.1 us, 8.8 split)
bool ColumnMeasured(const FcArgs& a) { return RingWindow(a) <= (a.m == 1 ? 4097 : 8193); }

bool FcW8RingSupported(const FcArgs& a) {
  if (!RingShapeOk(a) || a.ring_i_index < 0 || a.ring_o_index >= 0) return false;
  if (a.k > a.ring_size) return false;  // (the window stays within one turn of the ring)
  const int w_ks = DivUp(a.weights_k > 0 ? a.weights_k : a.k, 4);
  if (a.ring_size > 4 * w_ks || (a.weights_batch > 1 && a.ring_size != 4 * w_ks)) return false;
  return a.m <= 64 && (PartsSupported(a) || ColumnUs(a) <= UnspecialisedUs(a));
}

// Ring over the output channels.  Below 64 KB of weights a launch costs what a launch costs on either
// kernel, and the unspecialised one keeps those.
bool FcW8RingOSupported(const FcArgs& a) {
  if (!RingShapeOk(a) || a.ring_o_index < 0 || a.ring_i_index >= 0) return false;
  if (a.m > 64) return false;
  return (size_t)DivUp(a.k, 4) * DivUp(a.n, 4) * 16 >= 65536;
}

static RingParams MakeRingParams(const FcArgs& a) {
  RingParams p;
  p.act = a.act;
  p.weights = reinterpret_cast<const u32x4*>(a.weights);
  p.scale = a.scale;
  p.zero_point = a.has_zero_point ? a.zero_point : nullptr;
  p.bias = a.bias;
  p.dst = a.dst;
  p.partial = a.partial;
  p.params = a.params;
  p.batch_ids = a.batch_ids;
  p.m = a.m;
  p.ks = DivUp(a.k, 4);
  p.ns = DivUp(a.n, 4);
  p.ring_size = a.ring_size;
  p.ring_rows = a.ring_size / 4;
  p.ring_index = a.ring_i_index >= 0 ? a.ring_i_index : a.ring_o_index;
  p.src_end_ch_index = a.src_end_ch_index;
  p.dst_end_ch_index = a.dst_end_ch_index;
  p.k_channels = a.k;
  p.rows = a.rows;
  p.src_rows = a.src_rows;
  p.weights_batch = a.weights_batch;
  p.scale_kind = a.scale_kind;
  p.has_zero_point = a.has_zero_point ? 1 : 0;
  p.scalar_scale = a.scalar_scale;
  p.scalar_zero_point = a.scalar_zero_point;
  p.parts = 1;
  p.xcd_mask = p.xcd_runs = 0;
  return p;
}

hipError_t LaunchFcW8RingO(const FcArgs& a, hipStream_t stream, const char** kernel_name) {
  if (!FcW8RingOSupported(a)) return hipErrorInvalidValue;
  const RingParams p = MakeRingParams(a);
  if (kernel_name) *kernel_name = "fc_w8_ring_o_kernel";
  // every channel of the ring is a dst channel (and no runtime bound leaves some out)
  const bool turn = a.n == a.ring_size && p.dst_end_ch_index < 0;
  SetWhole(a.whole, turn);
  // token slots: as ColumnSlots (4 tokens x 8192 positions x 256 channels: 3.6 us with two, 3.9 with four; 8 tokens x 16384 x
  // 128: 4.2 against 4.1).  The turn kernel, whose start waits for less, has four ahead where two give every CU two work-groups: about half as
  // many.  (223 random turns of 4 .. 40 tokens with 256 .. 512 work-groups of four slots, speed over the other kernel with four / two slots:
  // whole fours of tokens or one less 1.11 .. 1.20 / 1.08 .. 1.09; one or two tokens more, where four slots leave two or three empty, below 384
  // work-groups 1.06 / 1.08 with 0.85 the least, from there on 1.13 / 1.08.)
  int slots = (turn ? (long)DivUp(p.ns, 16) * p.rows * DivUp(p.m, 2) : (long)DivUp(p.ns, 16) * p.rows * DivUp(p.m, 4)) >= 512 ? 4 : 2;
  while (slots > p.m) slots /= 2;
  SetTiles(a.tiles, slots, 4, 1);
  return a.act_f16 ? LaunchRingO<__half>(p, slots, turn, stream) : LaunchRingO<float>(p, slots, turn, stream);
}

hipError_t LaunchFcW8Ring(const FcArgs& a, hipStream_t stream, const char** kernel_name) {
  if (!FcW8RingSupported(a)) return hipErrorInvalidValue;
  RingParams p = MakeRingParams(a);
  if (kernel_name) *kernel_name = "fc_w8_ring_i_kernel";
  if (!PartsSupported(a) || (ColumnMeasured(a) && ColumnUs(a) <= SplitUs(a))) {
    const int slots = ColumnSlots(a);
    const bool small = RingWindow(a) <= 512;
    p.xcd_runs = std::min(8, DivUp(p.ns, 8));
    p.xcd_mask = p.xcd_runs == 1 ? 7 : (p.xcd_runs == 2 ? 3 : (p.xcd_runs <= 4 ? 1 : 0));
    SetVariant(a.variant, "column");
    const int turn = ColumnTurns(a, slots, small) ? (ColumnGroupsPerCu(a, slots, small) <= 1.0 ? 2 : 1) : 0;
    SetWhole(a.whole, turn > 0);
    SetTiles(a.tiles, slots, small ? 4 : 16, 1);
    return a.act_f16 ? LaunchColumn<__half>(p, slots, small, turn, stream) : LaunchColumn<float>(p, slots, small, turn, stream);
  }
  SetVariant(a.variant, "split");
  const RingSplit split = SplitWindow(a);
  SetTiles(a.tiles, a.m == 1 ? 1 : (a.m == 2 ? 2 : 4), kRingThreads / 64, split.parts);
  const int ls = split.lanes;
  p.parts = split.parts;
  if (a.act_f16) {
    if (ls == 16) return LaunchRingT<__half, 16>(p, a.dst_f16, stream);
    if (ls == 32) return LaunchRingT<__half, 32>(p, a.dst_f16, stream);
    return LaunchRingT<__half, 64>(p, a.dst_f16, stream);
  }
  if (ls == 16) return LaunchRingT<float, 16>(p, a.dst_f16, stream);
  if (ls == 32) return LaunchRingT<float, 32>(p, a.dst_f16, stream);
  return LaunchRingT<float, 64>(p, a.dst_f16, stream);
}

}  // namespace mldhip
