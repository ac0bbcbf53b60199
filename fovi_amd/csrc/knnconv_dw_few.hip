// Weight gradient of few-channel kNN-conv layers (c_in <= 8) from a bf16 output gradient:
// dW[o, c * V + v] = sum over images b and the (output n, input i) pairs of slot v of
// dy[b, n, o] * x[b, i, c], x fp32 or bf16.
//
// The images are the reduction index of the matrix instructions. A first pass lays both operands
// out in steps of 16 images (dyT[step][n][o][16], xT[step][i][c][16], bf16, padded with zero
// images), so that a lane loads its 8 images of one row or column with one 16-byte load, the rows of
// a point adjacent, and nothing passes through LDS (with all images of a row adjacent, [n][o][b],
// every lane pair read another line: 278 us for the products below). fp32 x is split into three
// bf16 parts by truncation (8 + 8 + 8 significant bits: exact), each multiplied with dy: the
// products are exact, the sums fp32, as in an fp32 product.
// A wave owns all rows o of a tile of up to 96 and a block of 32 columns, 32 / c_in slots x c_in
// channels; for every point of its range it reads the slots' neighbour lists, one neighbour of every
// slot per round (a slot without one reads a zero row), and skips a block none of whose slots has a
// neighbour. Partial tiles per point range go to a workspace and are added in range order.
// With a non-finite dy (a flag its layout pass sets) the waves form every point's slot sums and multiply
// those once, empty slots too, so that infinities and NaN come out as from the product of dy with
// the matrix of slot sums: inf times an empty slot's zero is NaN, times a non-zero sum inf.
// 128 images, 3 -> 96 channels, 4085 -> 964 points, k = 121 in V = 484 slots, x fp32: the slot-sum
// matrix (717 MB) and an fp32 GEMM over it took 650 + 643 us; here 151 us, 32 us for the layouts and
// 20 us for the reduction. Bound by the latency of the operand loads (two column blocks per wave, two
// waves per SIMD and no load ahead: 227 us).
#include <cmath>
#include <type_traits>

#include "common.h"

namespace fovi {
namespace {

typedef uint32_t u32x4f __attribute__((ext_vector_type(4)));

constexpr int DF_WAVES = 4;

// Three bf16 parts of v, large to small, by truncation: they add up to v exactly; a non-finite v is
// its own first part.
__device__ __forceinline__ void split3(float v, uint16_t (&part)[3]) {
  const uint32_t bits = __float_as_uint(v);
  const float h = __uint_as_float(bits & 0xffff0000u);
  const bool fin = (bits & 0x7f800000u) != 0x7f800000u;
  const float r1 = fin ? v - h : 0.0f;
  const float m = __uint_as_float(__float_as_uint(r1) & 0xffff0000u);
  uint32_t hi = bits >> 16;
  if (!fin && (bits & 0x007fffffu) && !(bits & 0x007f0000u)) hi |= 1u;   // NaN stays NaN
  part[0] = static_cast<uint16_t>(hi);
  part[1] = static_cast<uint16_t>(__float_as_uint(m) >> 16);
  part[2] = static_cast<uint16_t>(__float_as_uint(r1 - m) >> 16);
}

// ---- operands with the images adjacent ------------------------------------------------------
// out[((b / 16) * rows + fast * of + slow * os) * 16 + b % 16], `plane` elements apart for the parts;
// a block takes 64 fast indices of one slow index and 64 images through LDS: reads run along the
// fast dimension of the input, a thread writes 8 images of a row.
struct LayoutParams {
  const void* in;
  int64_t B, F, S, sb, sf, ss;           // images, fast and slow counts, their element strides
  uint16_t* out;
  int64_t of, os, rows, bp, plane;
  int32_t* flag;                         // set if a value is not finite (or NULL)
};

template <typename InT, int NS>
__global__ __launch_bounds__(256) void images_adjacent_kernel(LayoutParams p, uint32_t f_tiles, uint32_t b_tiles) {
  typedef typename std::conditional<std::is_same<InT, float>::value, float, uint16_t>::type T;
  __shared__ T tile[64][65];
  const uint32_t ft = blockIdx.x % f_tiles, rest = blockIdx.x / f_tiles;
  const int64_t f0 = static_cast<int64_t>(ft) * 64, b0 = static_cast<int64_t>(rest % b_tiles) * 64;
  const int64_t s = rest / b_tiles;
  const T* in = static_cast<const T*>(p.in) + s * p.ss;
  for (int k = threadIdx.x >> 6; k < 64; k += 4) {
    const int64_t f = f0 + (threadIdx.x & 63), b = b0 + k;
    tile[k][threadIdx.x & 63] = f < p.F && b < p.B ? in[b * p.sb + f * p.sf] : T(0);
  }
  __syncthreads();
  for (int k = threadIdx.x; k < 512; k += 256) {
    const int64_t f = f0 + (k & 63), b = b0 + 8 * (k >> 6);
    if (f >= p.F || b >= p.bp) continue;
    uint32_t part[NS][4];
#pragma unroll
    for (int q = 0; q < NS; ++q)
#pragma unroll
      for (int u = 0; u < 4; ++u) part[q][u] = 0u;
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const T v = tile[8 * (k >> 6) + u][k & 63];
      const int sh = (u & 1) * 16;
      if constexpr (NS == 1) {
        part[0][u >> 1] |= static_cast<uint32_t>(v) << sh;
        if (p.flag && (v & 0x7f80u) == 0x7f80u) *p.flag = 1;
      } else {
        uint16_t t[3];
        split3(v, t);
#pragma unroll
        for (int q = 0; q < NS; ++q) part[q][u >> 1] |= static_cast<uint32_t>(t[q]) << sh;
      }
    }
    uint16_t* o = p.out + ((b >> 4) * p.rows + f * p.of + s * p.os) * 16 + (b & 8);
#pragma unroll
    for (int q = 0; q < NS; ++q)
      *reinterpret_cast<u32x4f*>(o + q * p.plane) = u32x4f{part[q][0], part[q][1], part[q][2], part[q][3]};
  }
}

// the zero row (c_in x 16 values) of every step and part, and the flag
__global__ __launch_bounds__(128) void zero_rows_kernel(uint16_t* out, int count, int64_t step, int64_t plane, int ns,
                                                        int32_t* flag) {
  if (blockIdx.x == 0 && threadIdx.x == 0) *flag = 0;
  if (static_cast<int>(threadIdx.x) < count)
    for (int q = 0; q < ns; ++q) out[q * plane + blockIdx.x * step + threadIdx.x] = 0;
}

// ---- the products ------------------------------------------------------------------------------
struct DwFewParams {
  const uint16_t* dyt;                   // [bp / 16][n_out][c_out][16]
  const uint16_t* xt;                    // [parts][bp / 16][n_in + 1][c_in][16], row n_in zero
  int64_t plane;
  int C, Cout, Nin, Nout, V, K, bp;
  int slots;                             // slots per column block: 32 / c_in
  int n_ct, per;                         // column blocks, points per range
  const int32_t* slot_ptr;
  const int32_t* nbr;
  const int32_t* flag;                   // dy holds a non-finite value
  float* part;                           // [ranges][o tiles][n_ct][MB * 32][32]
};

template <int MB, int NS>
__global__ __launch_bounds__(DF_WAVES * 64, 3) void knnconv_dw_few_kernel(DwFewParams p, int ct_groups, int ranges) {
  const int lane = threadIdx.x & 63, h = lane >> 5, l32 = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lb = static_cast<int>(xcd_tile(blockIdx.x, gridDim.x));   // a range's column tiles share an L2
  const int ct = lb % ct_groups * DF_WAVES + wave;
  const int range = lb / ct_groups;
  if (range >= ranges) return;
  const int o0 = blockIdx.y * MB * 32;
  if (ct >= p.n_ct) return;              // no barrier follows
  int n0 = range * p.per;
  const int n1 = min(p.Nout, n0 + p.per);

  // this lane's column: slot v, channel c (columns past the slots: none)
  const int c = l32 % p.C, sl = l32 / p.C;
  int v = sl < p.slots ? ct * p.slots + sl : p.V;
  if (v >= p.V) v = -1;
  uint32_t oa[MB];                       // row offsets of dyT within a point
#pragma unroll
  for (int m = 0; m < MB; ++m) {
    const int o = min(o0 + m * 32 + l32, p.Cout - 1);
    oa[m] = static_cast<uint32_t>(o) * 16 + 8 * h;
  }

  f32x16 acc[MB];
#pragma unroll
  for (int m = 0; m < MB; ++m)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[m][r] = 0.0f;

  auto word = [&](int n) { return n < n1 && v >= 0 ? p.slot_ptr[static_cast<int64_t>(n) * p.V + v] : 0; };
  auto row = [&](int n, int w, int r) {  // the slot's r-th neighbour, or the zero row
    return r < (w & 0xffff) ? p.nbr[static_cast<int64_t>(n) * p.K + (w >> 16) + r] : p.Nin;
  };
  const int64_t dstep = static_cast<int64_t>(p.Nout) * p.Cout * 16, xstep = static_cast<int64_t>(p.Nin + 1) * p.C * 16;
  const int steps = p.bp / 16;
  struct Ops { bf16x8 a[MB], x[NS]; };
  if (*p.flag != 0) {
    // the slot sums (fp32, list order), then their parts; a zero part of a non-zero sum is replaced by
    // the smallest normal number of its sign, so that no part turns inf * sum into NaN
    for (int n = n0; n < n1; ++n) {
      const int w = word(n);
      const uint16_t* dn = p.dyt + static_cast<int64_t>(n) * p.Cout * 16;
      for (int s = 0; s < steps; ++s) {
        float sum[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) sum[u] = 0.0f;
        for (int r = 0; __builtin_amdgcn_ballot_w64((w & 0xffff) > r) != 0; ++r) {
          const uint16_t* xr = p.xt + (static_cast<int64_t>(row(n, w, r)) * p.C + c) * 16 + 8 * h + s * xstep;
          float x[8];
#pragma unroll
          for (int q = 0; q < NS; ++q)
#pragma unroll
            for (int u = 0; u < 8; ++u) {          // large parts first: exact
              const float t = bf16_bits_to_f32(xr[q * p.plane + u]);
              x[u] = q == 0 ? t : x[u] + t;
            }
#pragma unroll
          for (int u = 0; u < 8; ++u) sum[u] += x[u];
        }
        bf16x8 xs[NS];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          if constexpr (NS == 1) {
            xs[0][u] = static_cast<__bf16>(sum[u]);
          } else {
            uint16_t part[3];
            split3(sum[u], part);
#pragma unroll
            for (int q = 0; q < NS; ++q) {
              if ((part[q] & 0x7fffu) == 0u && sum[u] != 0.0f)
                part[q] = 0x0080u | (__float_as_uint(sum[u]) >> 31 << 15);
              xs[q][u] = __builtin_bit_cast(__bf16, part[q]);
            }
          }
        }
#pragma unroll
        for (int m = 0; m < MB; ++m) {
          const bf16x8 a = *reinterpret_cast<const bf16x8*>(dn + s * dstep + oa[m]);
#pragma unroll
          for (int q = NS - 1; q >= 0; --q) acc[m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, xs[q], acc[m], 0, 0, 0);
        }
      }
    }
    n0 = n1;
  }
  int w = word(n0), i0 = n0 < n1 ? row(n0, w, 0) : p.Nin, wn = word(n0 + 1);
  for (int n = n0; n < n1; ++n) {
    // the next point's first neighbours, the one after's words
    const int inx = n + 1 < n1 ? row(n + 1, wn, 0) : p.Nin, wnn = word(n + 2);
    const uint16_t* dn = p.dyt + static_cast<int64_t>(n) * p.Cout * 16;
    for (int r = 0; __builtin_amdgcn_ballot_w64((w & 0xffff) > r) != 0; ++r) {
      const int i = r == 0 ? i0 : row(n, w, r);
      const uint16_t* xr = p.xt + (static_cast<int64_t>(i) * p.C + c) * 16 + 8 * h;
      auto fetch = [&](Ops& t, int s) {
#pragma unroll
        for (int m = 0; m < MB; ++m) t.a[m] = *reinterpret_cast<const bf16x8*>(dn + s * dstep + oa[m]);
#pragma unroll
        for (int q = 0; q < NS; ++q) t.x[q] = *reinterpret_cast<const bf16x8*>(xr + s * xstep + q * p.plane);
      };
      auto multiply = [&](const Ops& t) {
#pragma unroll
        for (int q = NS - 1; q >= 0; --q)          // small parts first
#pragma unroll
          for (int m = 0; m < MB; ++m) acc[m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(t.a[m], t.x[q], acc[m], 0, 0, 0);
      };
      // the next 16 images' operands are loaded while these are multiplied (the last step loads
      // its own again: a conditional load would make every wait a full one)
      Ops t0, t1;
      fetch(t0, 0);
      for (int s = 0;;) {
        int nx = min(s + 1, steps - 1);
        fetch(t1, nx);
        multiply(t0);
        if (nx == s) break;
        s = nx;
        nx = min(s + 1, steps - 1);
        fetch(t0, nx);
        multiply(t1);
        if (nx == s) break;
        s = nx;
      }
    }
    w = wn; wn = wnn; i0 = inx;
  }
  float* out = p.part + ((static_cast<int64_t>(range) * gridDim.y + blockIdx.y) * p.n_ct + ct) * (MB * 32 * 32);
#pragma unroll
  for (int m = 0; m < MB; ++m)
#pragma unroll
    for (int r = 0; r < 16; ++r) out[(m * 32 + 8 * (r >> 2) + 4 * h + (r & 3)) * 32 + l32] = acc[m][r];
}

__global__ __launch_bounds__(256) void knnconv_dw_few_reduce_kernel(DwFewParams p, int mb, int ranges, int o_tiles,
                                                                    float* dw) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (t >= static_cast<int64_t>(p.Cout) * p.C * p.V) return;
  const int v = static_cast<int>(t % p.V);
  const int c = static_cast<int>((t / p.V) % p.C), o = static_cast<int>(t / (static_cast<int64_t>(p.V) * p.C));
  const int blk = v / p.slots, col = (v % p.slots) * p.C + c;
  const int rows = mb * 32;
  const float* src = p.part + (static_cast<int64_t>(o / rows) * p.n_ct + blk) * (rows * 32) + (o % rows) * 32 + col;
  const int64_t stride = static_cast<int64_t>(o_tiles) * p.n_ct * rows * 32;
  float sum = 0.0f;
  int s = 0;
  for (; s + 8 <= ranges; s += 8) {
    float x[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) x[u] = src[(s + u) * stride];
#pragma unroll
    for (int u = 0; u < 8; ++u) sum += x[u];
  }
  for (; s < ranges; ++s) sum += src[s * stride];
  dw[t] = sum;
}

struct FewPlan {
  int64_t bp, dyt, xt, part;             // images padded; elements of dyT, xT (a part), partials
  int parts, slots, n_ct, mb, o_tiles, ranges, per;
};

bool few_plan(int64_t B, int64_t C, int64_t Cout, int64_t Nin, int64_t Nout, int64_t V, int x_dtype, FewPlan& f) {
  if (B < 1 || C < 1 || C > 8 || Cout < 1 || Nin < 1 || Nout < 1 || V < 1 || (x_dtype != FOVI_F32 && x_dtype != FOVI_BF16))
    return false;
  constexpr int64_t lim = int64_t(1) << 31;
  f.bp = (B + 15) / 16 * 16;
  if (f.bp >= (1 << 20) || Cout >= (1 << 20) || Nin >= lim - 1 || Nout >= lim || V >= (1 << 20) || Cout * f.bp >= lim || Cout * 16 >= lim)
    return false;
  f.parts = x_dtype == FOVI_F32 ? 3 : 1;
  f.slots = static_cast<int>(32 / C);
  f.n_ct = static_cast<int>((V + f.slots - 1) / f.slots);
  // tiles of up to 96 rows (accumulators and two steps' operands for three waves per SIMD), as even
  // as they come
  const int64_t row_blocks = (Cout + 31) / 32;
  f.o_tiles = static_cast<int>((row_blocks + 2) / 3);
  f.mb = static_cast<int>((row_blocks + f.o_tiles - 1) / f.o_tiles);
  // point ranges: about 3072 waves in all (three per SIMD), each range at least one point. A wave's
  // chain takes about a microsecond per point and step of 16 images, the reduction's 75 ns per range
  // (eight loads in flight), so their sum is least at sqrt(13 steps points) ranges: more only
  // lengthen the reduction (1156 points, 8 images, one tile: 89 us with 1156 ranges, 40 with 122).
  const int64_t tiles = static_cast<int64_t>(f.n_ct) * f.o_tiles;
  int64_t ranges = 3072 / tiles > 0 ? 3072 / tiles : 1;
  if (ranges > Nout) ranges = Nout;
  const double chain = std::sqrt(13.0 * static_cast<double>(f.bp / 16) * static_cast<double>(Nout));
  if (ranges > chain) ranges = static_cast<int64_t>(chain);
  const int64_t per = (Nout + ranges - 1) / ranges;
  f.per = static_cast<int>(per);
  f.ranges = static_cast<int>((Nout + per - 1) / per);
  f.dyt = (Nout * Cout * f.bp + 63) / 64 * 64;
  f.xt = ((Nin + 1) * C * f.bp + 63) / 64 * 64;
  f.part = static_cast<int64_t>(f.ranges) * tiles * f.mb * 32 * 32;
  return true;
}

template <typename InT, int NS>
int lay_out(const void* in, int64_t B, int64_t C, int64_t N, const int64_t* st, uint16_t* out, int64_t out_rows,
            int64_t bp, int64_t plane, int32_t* flag, hipStream_t s) {
  LayoutParams p;
  p.in = in; p.B = B; p.sb = st[0]; p.out = out; p.bp = bp; p.plane = plane; p.rows = out_rows; p.flag = flag;
  const bool rows = st[1] == 1 && C > 1;         // channels adjacent: they are the fast dimension
  p.F = rows ? C : N; p.S = rows ? N : C;
  p.sf = rows ? st[1] : st[2]; p.ss = rows ? st[2] : st[1];
  p.of = rows ? 1 : C; p.os = rows ? C : 1;      // row n * C + c
  const int64_t ft = (p.F + 63) / 64, bt = (bp + 63) / 64;
  if (ft * bt * p.S > 0x7fffffffLL) { set_error("fovi_knnconv_dw_few: too large"); return 1; }
  hipLaunchKernelGGL((images_adjacent_kernel<InT, NS>), dim3(static_cast<unsigned>(ft * bt * p.S)), dim3(256), 0, s, p,
                     static_cast<uint32_t>(ft), static_cast<uint32_t>(bt));
  return check_launch("fovi_knnconv_dw_few(layout)");
}

template <int NS>
int launch_few(const DwFewParams& p, const FewPlan& f, hipStream_t s) {
  const int groups = (f.n_ct + DF_WAVES - 1) / DF_WAVES;
  const dim3 grid(static_cast<unsigned>((static_cast<int64_t>(groups) * f.ranges + 7) / 8 * 8), static_cast<unsigned>(f.o_tiles));
  const auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(DF_WAVES * 64), 0, s, p, groups, f.ranges); };
  if (f.mb == 1) go(knnconv_dw_few_kernel<1, NS>);
  else if (f.mb == 2) go(knnconv_dw_few_kernel<2, NS>);
  else go(knnconv_dw_few_kernel<3, NS>);
  return check_launch("fovi_knnconv_dw_few");
}

}  // namespace
}  // namespace fovi

extern "C" int64_t fovi_knnconv_dw_few_workspace_bytes(int64_t batch, int64_t c_in, int64_t c_out, int64_t n_in,
                                                       int64_t n_out, int64_t n_ref, int32_t x_dtype) {
  fovi::FewPlan f;
  if (!fovi::few_plan(batch, c_in, c_out, n_in, n_out, n_ref, x_dtype, f)) return -1;
  return (f.dyt + f.parts * f.xt) * 2 + f.part * 4 + 16;
}

// Microseconds on the plan above, fitted to 5288 calls (1 to 8 channels, 8 to 384 outputs, 4 to 16384
// points, V = 9 to 484, 1 to 128 images; estimate / time: 0.65 to 1.3 for 98% of them): launches, a wave's
// chain over its points, the layout passes (0.6 us per MB read and written), the partial tiles.
extern "C" double fovi_knnconv_dw_few_us(int64_t batch, int64_t c_in, int64_t c_out, int64_t n_in, int64_t n_out,
                                         int64_t n_ref, int32_t x_dtype, double rounds) {
  fovi::FewPlan f;
  if (!fovi::few_plan(batch, c_in, c_out, n_in, n_out, n_ref, x_dtype, f)) return -1.0;
  const double chain = f.per * rounds, steps = static_cast<double>(f.bp / 16);
  const double layout = static_cast<double>(n_out) * c_out * (batch + f.bp) * 2 +
                        static_cast<double>(n_in) * c_in * ((f.parts == 3 ? 4 : 2) * batch + 2 * f.parts * f.bp);
  return 15.0 + 0.2 * chain + (f.parts == 3 ? 0.65 : 0.45) * chain * steps + 0.6e-6 * layout +
         0.43e-6 * static_cast<double>(f.part) * 8 + 0.02 * f.ranges;
}

extern "C" int fovi_knnconv_dw_few(const fovi_knnconv_dw_few_args* a, void* stream) {
  using namespace fovi;
  clear_error();
  if (!a || !a->x || !a->dy || !a->slot_ptr || !a->nbr_sorted || !a->workspace || !a->dw) {
    set_error("fovi_knnconv_dw_few: null pointer");
    return 1;
  }
  FewPlan f;
  if (a->k < 1 || a->k > 32767 || !few_plan(a->batch, a->c_in, a->c_out, a->n_in, a->n_out, a->n_ref, a->x_dtype, f)) {
    set_error("fovi_knnconv_dw_few: bad sizes (1 to 8 input channels, F32 or BF16 input)");
    return 1;
  }
  const int64_t need = (f.dyt + f.parts * f.xt) * 2 + f.part * 4 + 16;
  if (a->workspace_bytes < need || reinterpret_cast<uintptr_t>(a->workspace) % 16 != 0) {
    set_error("fovi_knnconv_dw_few: workspace %lld bytes (16-byte aligned), need %lld", (long long)a->workspace_bytes,
              (long long)need);
    return 1;
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  DwFewParams p;
  float* part = static_cast<float*>(a->workspace);             // a multiple of 128 bytes
  uint16_t* dyt = reinterpret_cast<uint16_t*>(part + f.part);
  uint16_t* xt = dyt + f.dyt;
  int32_t* flag = reinterpret_cast<int32_t*>(xt + f.parts * f.xt);
  const int64_t x_rows = (a->n_in + 1) * a->c_in;
  hipLaunchKernelGGL(zero_rows_kernel, dim3(static_cast<unsigned>(f.bp / 16)), dim3(128), 0, s,
                     xt + a->n_in * a->c_in * 16, static_cast<int>(a->c_in) * 16, x_rows * 16, f.xt, f.parts, flag);
  if (check_launch("fovi_knnconv_dw_few(zero row)")) return 1;
  if (lay_out<uint16_t, 1>(a->dy, a->batch, a->c_out, a->n_out, a->dy_stride, dyt, a->n_out * a->c_out, f.bp, 0, flag, s)) return 1;
  if (a->x_dtype == FOVI_F32 ? lay_out<float, 3>(a->x, a->batch, a->c_in, a->n_in, a->x_stride, xt, x_rows, f.bp, f.xt, nullptr, s)
                             : lay_out<uint16_t, 1>(a->x, a->batch, a->c_in, a->n_in, a->x_stride, xt, x_rows, f.bp, f.xt,
                                                    nullptr, s))
    return 1;
  p.dyt = dyt; p.xt = xt; p.plane = f.xt;
  p.C = static_cast<int>(a->c_in); p.Cout = static_cast<int>(a->c_out); p.Nin = static_cast<int>(a->n_in);
  p.Nout = static_cast<int>(a->n_out); p.V = static_cast<int>(a->n_ref); p.K = static_cast<int>(a->k);
  p.bp = static_cast<int>(f.bp); p.slots = f.slots; p.n_ct = f.n_ct; p.per = f.per;
  p.slot_ptr = a->slot_ptr; p.nbr = a->nbr_sorted; p.flag = flag; p.part = part;
  if (f.parts == 3 ? launch_few<3>(p, f, s) : launch_few<1>(p, f, s)) return 1;
  const int64_t n = a->c_out * a->c_in * a->n_ref;
  hipLaunchKernelGGL(knnconv_dw_few_reduce_kernel, dim3(static_cast<unsigned>((n + 255) / 256)), dim3(256), 0, s, p, f.mb,
                     f.ranges, f.o_tiles, a->dw);
  return check_launch("fovi_knnconv_dw_few(reduce)");
}
