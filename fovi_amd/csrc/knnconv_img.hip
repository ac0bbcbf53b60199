// kNN-convolution forward with image rows: fp32, bf16 and e4m3 layers whose batch is large
// enough that the rows of a matrix block are images of one output point (or of a few).
//
// GEMM view: rows = (output point, image), columns = output channels, reduction = (slot v,
// channel c). Only the slots in which a point has a neighbour contribute: on the log-polar
// lattice with k = V = 25 a point uses 16 of its 25 slots, with a doubled ref grid (V = 100)
// 23 of 100. The kernels whose tiles are 256 points of one image visit every slot, since some
// point of the tile uses it. Here a workgroup owns PP points x IB images (PP * IB = 32 RB rows)
// and visits only the union of its points' slots:
//  * the host table (fovi_knnconv_img_tables) puts points with similar slot sets into a group,
//    within windows of consecutive points, and lists the group's slots in the layer's slot
//    visit order: per (slot, point) the first two neighbours, the count and the list start;
//  * the reduction runs over 64-byte channel chunks (outer) and the group's slots (inner). Every
//    thread gathers 16-byte parts of the input rows of the next two (chunk, slot) stages while
//    the matrix units work on the current two, sums them where a slot has several neighbours
//    (fp32, list order, rounded once), and writes them to LDS (64-byte rows, XOR-swizzled);
//  * weights come from global memory in fragment order straight into registers; the 4 waves of
//    a workgroup own disjoint columns, so each fragment is loaded once per workgroup;
//  * two workgroups share a CU (two waves per SIMD), so one's gathers and sums run beside the
//    other's MFMAs.
// A skipped slot would have added products of zeros: +0 to an accumulator that is never -0, so
// for finite weights the outputs are those of the kernels that visit every slot in the same
// order, bit for bit. With a non-finite packed weight (the flag that packing writes) every slot
// of the list is visited, the unused ones too (0 * inf is NaN).
#include <algorithm>
#include <thread>
#include <type_traits>
#include <vector>

#include "knnconv_internal.h"

namespace fovi {

namespace {

constexpr int IM_WAVES = 4;
constexpr int IM_THREADS = IM_WAVES * 64;
constexpr uint32_t IM_NONE = 0x80000000u;   // past every buffer's range: reads zeros

typedef int i32x8i __attribute__((ext_vector_type(8)));
typedef uint32_t u32x8i __attribute__((ext_vector_type(8)));
typedef float f32x16s __attribute__((ext_vector_type(16)));

// Table memory no kernel writes: constant address space, so that uniform reads are scalar loads.
template <typename T> using Const = const __attribute__((address_space(4))) T;
template <typename T> __device__ __forceinline__ Const<T>* as_const(const T* ptr) {
  return (Const<T>*)ptr;
}

struct ImgTables {
  const u32x4* ent;       // [groups, V, PP]: neighbours 1 and 2, count << 16 | begin, position
  const int32_t* points;  // [groups, PP] output point (-1: none)
  const int32_t* nact;    // [groups] slots of the union
  const int32_t* flag;    // non-zero: a packed weight is not finite
  int64_t groups;
  int pp, ib, ibs;        // points and images per group row block; log2(ib)
  int ncb;                // 32-column blocks of the packed weight
};

// Element types. A 64-byte LDS row is one chunk of CH channels, a 16-byte part PC channels.
template <int DT> struct ImElem;
template <> struct ImElem<FOVI_BF16> {
  static constexpr int ES = 2, CH = 32, PC = 8;
  typedef f32x8 Sum;
  static __device__ __forceinline__ Sum first(u32x4 x) { return unpack_bf16x8(x); }
  static __device__ __forceinline__ void add(Sum& a, u32x4 x) { a += unpack_bf16x8(x); }
  static __device__ __forceinline__ u32x4 pack(const Sum& a) {
    return u32x4{cvt_pk_bf16(a[0], a[1]), cvt_pk_bf16(a[2], a[3]), cvt_pk_bf16(a[4], a[5]), cvt_pk_bf16(a[6], a[7])};
  }
};
template <> struct ImElem<FOVI_F32> {
  static constexpr int ES = 4, CH = 16, PC = 4;
  typedef f32x4 Sum;
  static __device__ __forceinline__ Sum first(u32x4 x) { return __builtin_bit_cast(f32x4, x); }
  static __device__ __forceinline__ void add(Sum& a, u32x4 x) { a += __builtin_bit_cast(f32x4, x); }
  static __device__ __forceinline__ u32x4 pack(const Sum& a) { return __builtin_bit_cast(u32x4, a); }
};
template <> struct ImElem<FOVI_F8E4M3> {
  static constexpr int ES = 1, CH = 64, PC = 16;
  typedef f32x16s Sum;
  static __device__ __forceinline__ Sum first(u32x4 x) {
    Sum s;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const auto lo = __builtin_amdgcn_cvt_pk_f32_fp8(static_cast<int>(x[w]), false);
      const auto hi = __builtin_amdgcn_cvt_pk_f32_fp8(static_cast<int>(x[w]), true);
      s[4 * w] = lo[0]; s[4 * w + 1] = lo[1]; s[4 * w + 2] = hi[0]; s[4 * w + 3] = hi[1];
    }
    return s;
  }
  static __device__ __forceinline__ void add(Sum& a, u32x4 x) { a += first(x); }
  static __device__ __forceinline__ u32x4 pack(const Sum& a) {
    u32x4 out;
#pragma unroll
    for (int w = 0; w < 4; ++w)
      out[w] = cvt_pk_e4m3<true>(a[4 * w + 2], a[4 * w + 3],
                                 cvt_pk_e4m3<false>(a[4 * w], a[4 * w + 1], __float_as_uint(a[4 * w])));
    return out;
  }
};

// XOR pattern of the 16-byte parts of LDS row r (as swz32 in knnconv_internal.h)
__device__ __forceinline__ int im_swz(int r) { return (((r >> 1) ^ (r >> 3)) & 1) | ((r >> 1) & 2); }

// RB: 32-row blocks per workgroup; CB: 32-column blocks per wave. 16 consecutive rows are images of
// one point (ib >= 16), so the table entries a wave gathers by are uniform.
template <int DT, int RB, int CB>
__global__ __launch_bounds__(IM_THREADS, 2) void knnconv_img_kernel(KnnParams p, ImgTables t, int n_ct, int64_t total,
                                                                   int64_t padded, int vec_out) {
  typedef ImElem<DT> E;
  typedef typename E::Sum Sum;
  constexpr int M = RB * 32;
  constexpr int J = RB >= 2 ? RB / 2 : 1;          // rows per thread and stage
  constexpr int A_BYTES = M * 64;                  // one stage
  constexpr bool F32 = DT == FOVI_F32;
  constexpr int OPP = F32 ? 4 : 8;                 // outputs per 16-byte store
  constexpr int OES = F32 ? 4 : 2;
  constexpr int EW = CB * 32 + OPP;                // padded LDS row of the epilogue (elements)
  constexpr int E_BYTES = IM_WAVES * 32 * EW * OES;
  constexpr int S_BYTES = 4 * A_BYTES > E_BYTES ? 4 * A_BYTES : E_BYTES;
  __shared__ __attribute__((aligned(16))) uint8_t smem[S_BYTES];
  // the group's points (at most 128 / 16): written by the first wave, read by all in the epilogue,
  // with a barrier between on every path
  __shared__ int32_t s_pts[8];

  const int64_t lb = xcd_tile(blockIdx.x, padded);
  if (lb >= total) return;
  const int ct = static_cast<int>(lb % n_ct);
  const int64_t rest = lb / n_ct;
  const int64_t g = rest % t.groups;
  const int64_t img0 = (rest / t.groups) * t.ib;
  const int nimg = static_cast<int>(min(static_cast<int64_t>(t.ib), p.B - img0));
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int V = static_cast<int>(p.V);
  const int nact = *as_const(t.flag) ? V : as_const(t.nact)[g];
  const int nchan = static_cast<int>(p.C);
  const int nch = static_cast<int>((p.C + E::CH - 1) / E::CH);
  const int nst = nact * nch;
  const int cb0 = (ct * IM_WAVES + wave) * CB;
  const bool live = cb0 * 32 < p.Cout;             // the wave has columns (uniform)
  if (tid < t.pp) s_pts[tid] = t.points[g * t.pp + tid];

  // input rows of this block's images; the range check reads zeros past them
  const uint32_t row_b = static_cast<uint32_t>(p.xs2) * E::ES;
  const uint32_t img_b = static_cast<uint32_t>(p.xs0) * E::ES;
  const uint32_t range = static_cast<uint32_t>(nimg - 1) * img_b + static_cast<uint32_t>(p.Nin - 1) * row_b +
                         static_cast<uint32_t>(p.C) * E::ES;
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<char*>(static_cast<const char*>(p.x) + img0 * p.xs0 * E::ES), static_cast<short>(0),
      static_cast<int>(range), 0x00020000);

  // gather role: part q of rows r0 + 64 j (RB = 1: the waves take turns, two per stage)
  const int q = tid & 3;
  const int r0 = RB == 1 ? (tid & 127) >> 2 : tid >> 2;
  uint32_t voff[J];                                // the image's offset, IM_NONE past the batch
  int pj[J];                                       // the rows' point within the group (uniform)
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int r = r0 + 64 * j;
    const int i = r & (t.ib - 1);
    pj[j] = __builtin_amdgcn_readfirstlane(r >> t.ibs);
    voff[j] = i < nimg ? static_cast<uint32_t>(i) * img_b + q * 16 : IM_NONE;
  }

  Const<u32x4>* ent = as_const(t.ent) + g * V * t.pp;

  // the stage to gather next: slot gs of the group's list, chunk gc
  int gs = 0, gc = 0, gf = 0;
  struct Stage { u32x4 e[J]; uint32_t cofs; int pos, c; };
  // table entries of stage gf (no neighbours past the last), then on to the next
  auto fetch = [&](Stage& s) {
    const bool in = gf < nst;
    const int row = (in ? gs : 0) * t.pp;
#pragma unroll
    for (int j = 0; j < J; ++j) s.e[j] = ent[row + pj[j]];
    s.pos = in ? static_cast<int>(s.e[0][3]) : 0;
    s.c = in ? gc : 0;
    if (!in)
#pragma unroll
      for (int j = 0; j < J; ++j) { s.e[j][0] = IM_NONE; s.e[j][2] = 0u; }
    ++gf;
    if (++gs == nact) { gs = 0; ++gc; }
  };
  auto rowofs = [&](uint32_t n) { return n & IM_NONE ? IM_NONE : n * row_b; };
  // byte offset of the chunk, past the range for parts beyond the channels
  auto chunk_ofs = [&](int c) -> uint32_t {
    return c * E::CH + q * E::PC < nchan ? static_cast<uint32_t>(c) * 64u : IM_NONE;
  };
  // the sum of three offsets, past the range if any of them is (two IM_NONE would wrap round)
  auto sum_ofs = [&](uint32_t a, uint32_t b, uint32_t c) { return ((a | b | c) & IM_NONE) ? IM_NONE : a + b + c; };
  auto load = [&](uint32_t o) { return __builtin_amdgcn_raw_buffer_load_b128(rs, o, 0, 0); };
  auto issue = [&](Stage& s, u32x4 (&v0)[J], u32x4 (&v1)[J]) {
    s.cofs = chunk_ofs(s.c);
#pragma unroll
    for (int j = 0; j < J; ++j) v0[j] = load(sum_ofs(voff[j], rowofs(s.e[j][0]), s.cofs));
#pragma unroll
    for (int j = 0; j < J; ++j)
      if ((s.e[j][2] >> 16) > 1u) v1[j] = load(sum_ofs(voff[j], rowofs(s.e[j][1]), s.cofs));
  };
  auto finish = [&](const Stage& s, const u32x4 (&v0)[J], const u32x4 (&v1)[J], uint8_t* A) {
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const int r = r0 + 64 * j;
      u32x4 out = v0[j];
      const uint32_t cnt = s.e[j][2] >> 16;
      if (cnt > 1u) {
        Sum a = E::first(v0[j]);
        E::add(a, v1[j]);
        if (cnt > 2u) {
          Const<int32_t>* list = as_const(p.nbr) +
                                 static_cast<int64_t>(as_const(t.points)[g * t.pp + pj[j]]) * p.K +
                                 (s.e[j][2] & 0xffffu);
          uint32_t k = 2;
          for (; k + 1 < cnt; k += 2) {            // two rows in flight
            const u32x4 x0 = load(sum_ofs(voff[j], rowofs(static_cast<uint32_t>(list[k])), s.cofs));
            const u32x4 x1 = load(sum_ofs(voff[j], rowofs(static_cast<uint32_t>(list[k + 1])), s.cofs));
            E::add(a, x0);
            E::add(a, x1);
          }
          if (k < cnt) E::add(a, load(sum_ofs(voff[j], rowofs(static_cast<uint32_t>(list[k])), s.cofs)));
        }
        out = E::pack(a);
      }
      *reinterpret_cast<u32x4*>(A + r * 64 + ((q ^ im_swz(r)) << 4)) = out;
    }
  };

  // weight fragments of a stage: 2 * CB KB per wave
  const u32x4* wbase = static_cast<const u32x4*>(p.w) + static_cast<int64_t>(live ? cb0 : 0) * 128 + lane;
  auto load_w = [&](int pos, int c, u32x4 (&w)[CB * 2]) {
    const u32x4* src = wbase + (static_cast<int64_t>(c) * V + pos) * t.ncb * 128;
#pragma unroll
    for (int b = 0; b < CB * 2; ++b) w[b] = src[b * 64];
  };

  f32x16 acc[RB][CB];
#pragma unroll
  for (int i = 0; i < RB; ++i)
#pragma unroll
    for (int b = 0; b < CB; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][b][r] = 0.0f;

  const int lrow = (lane & 31) * 64, lg = im_swz(lane & 31), lh = lane >> 5;
  auto part = [&](const uint8_t* A, int i, int qq) {
    return *reinterpret_cast<const u32x4*>(A + i * 2048 + lrow + ((qq ^ lg) << 4));
  };
  auto compute = [&](const uint8_t* A, const u32x4 (&w)[CB * 2]) {
    if constexpr (DT == FOVI_F8E4M3) {
#pragma unroll
      for (int i = 0; i < RB; ++i) {
        const u32x4 a0 = part(A, i, 2 * lh), a1 = part(A, i, 2 * lh + 1);
        const i32x8i a8 = __builtin_bit_cast(i32x8i, u32x8i{a0[0], a0[1], a0[2], a0[3], a1[0], a1[1], a1[2], a1[3]});
#pragma unroll
        for (int b = 0; b < CB; ++b) {
          const u32x4 b0 = w[b * 2], b1 = w[b * 2 + 1];
          const i32x8i b8 = __builtin_bit_cast(i32x8i, u32x8i{b0[0], b0[1], b0[2], b0[3], b1[0], b1[1], b1[2], b1[3]});
          acc[i][b] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a8, b8, acc[i][b], 0, 0, 0, 127, 0, 127);
        }
      }
    } else {
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        u32x4 a[RB];
#pragma unroll
        for (int i = 0; i < RB; ++i) a[i] = part(A, i, 2 * ks + lh);
#pragma unroll
        for (int i = 0; i < RB; ++i)
#pragma unroll
          for (int b = 0; b < CB; ++b) {
            if constexpr (F32) {
              const f32x4 av = __builtin_bit_cast(f32x4, a[i]), wv = __builtin_bit_cast(f32x4, w[b * 2 + ks]);
#pragma unroll
              for (int e = 0; e < 4; ++e)
                acc[i][b] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[e], wv[e], acc[i][b], 0, 0, 0);
            } else {
              acc[i][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a[i]),
                                                                  __builtin_bit_cast(bf16x8, w[b * 2 + ks]),
                                                                  acc[i][b], 0, 0, 0);
            }
          }
      }
    }
  };
  auto barrier = [&]() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  };
  // An iteration multiplies two stages while the rows of the next two are gathered into registers,
  // and writes those to LDS at its end; the table entries are read one iteration further ahead.
  Stage cur[2], nxt[2];
  u32x4 v0[2][J], v1[2][J], wa[CB * 2], wb[CB * 2];
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int j = 0; j < J; ++j) { v0[s][j] = u32x4{0u, 0u, 0u, 0u}; v1[s][j] = u32x4{0u, 0u, 0u, 0u}; }
  const int half = wave >> 1;                      // RB = 1: the stage these waves gather
  auto gather = [&](Stage (&s)[2]) {
    if constexpr (RB > 1) { issue(s[0], v0[0], v1[0]); issue(s[1], v0[1], v1[1]); }
    else if (half == 0) issue(s[0], v0[0], v1[0]);
    else issue(s[1], v0[0], v1[0]);
  };
  auto deliver = [&](const Stage (&s)[2], int buf) {
    uint8_t* A = smem + buf * 2 * A_BYTES;
    if constexpr (RB > 1) { finish(s[0], v0[0], v1[0], A); finish(s[1], v0[1], v1[1], A + A_BYTES); }
    else if (half == 0) finish(s[0], v0[0], v1[0], A);
    else finish(s[1], v0[0], v1[0], A + A_BYTES);
  };
  if (nst > 0) {
    fetch(cur[0]); fetch(cur[1]);
    gather(cur);
    load_w(cur[0].pos, cur[0].c, wa);
    fetch(nxt[0]); fetch(nxt[1]);
    deliver(cur, 0);
    barrier();
    int pos1 = cur[1].pos, c1 = cur[1].c;
    const int ni = (nst + 1) / 2;
    for (int it = 0; it < ni; ++it) {
      const uint8_t* A = smem + (it & 1) * 2 * A_BYTES;
      if (live) load_w(pos1, c1, wb);
      gather(nxt);
      cur[0] = nxt[0]; cur[1] = nxt[1];
      fetch(nxt[0]); fetch(nxt[1]);
      if (live) {
        compute(A, wa);
        load_w(cur[0].pos, cur[0].c, wa);
        if (2 * it + 1 < nst) compute(A + A_BYTES, wb);
      }
      deliver(cur, (it & 1) ^ 1);
      pos1 = cur[1].pos; c1 = cur[1].c;
      barrier();
    }
  } else {
    barrier();   // a group none of whose points has a neighbour: s_pts, which every wave reads below
  }
  if (!live) return;

  // y = acc + bias (x_scale * w_scale[o] * acc + bias for e4m3), ReLU optional
  float bo[CB], sc[CB];
  const float xs = DT == FOVI_F8E4M3 ? (p.x_scale_dev ? *p.x_scale_dev : p.x_scale) : 1.0f;
#pragma unroll
  for (int b = 0; b < CB; ++b) {
    const int64_t o = (cb0 + b) * 32 + (lane & 31);
    bo[b] = (p.bias && o < p.Cout) ? p.bias[o] : 0.0f;
    sc[b] = DT == FOVI_F8E4M3 && o < p.Cout ? xs * p.w_scale[o] : 1.0f;
  }
  auto out_val = [&](float a, int b) {
    return epilogue(DT == FOVI_F8E4M3 ? a * sc[b] + bo[b] : a + bo[b], p.relu);
  };
  typedef typename std::conditional<F32, float, uint16_t>::type OutT;
  OutT* y = static_cast<OutT*>(p.y);
  auto row_ptr = [&](int r, bool& ok) -> OutT* {
    const int i = r & (t.ib - 1);
    const int32_t n = s_pts[r >> t.ibs];
    ok = i < nimg && n >= 0;
    return y + (img0 + i) * p.ys0 + static_cast<int64_t>(n) * p.ys2;
  };
  if (vec_out) {
    // each wave transposes its 32-row blocks through LDS and stores 16-byte pieces
    OutT* Eo = reinterpret_cast<OutT*>(smem) + wave * 32 * EW;
    constexpr int PPR = CB * 32 / OPP;            // 16-byte pieces per row
#pragma unroll
    for (int i = 0; i < RB; ++i) {
#pragma unroll
      for (int b = 0; b < CB; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          Elem<OutT>::store(&Eo[(8 * (r >> 2) + 4 * lh + (r & 3)) * EW + b * 32 + (lane & 31)], out_val(acc[i][b][r], b));
      __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0): this wave's LDS writes are done
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int k = 0; k < 32 * PPR / 64; ++k) {
        const int piece = k * 64 + lane;
        const int row = piece / PPR, pt = piece % PPR;
        const u32x4 val = *reinterpret_cast<const u32x4*>(&Eo[row * EW + pt * OPP]);
        bool ok;
        OutT* dst = row_ptr(i * 32 + row, ok);
        const int64_t o = cb0 * 32 + pt * OPP;
        if (ok && o < p.Cout) *reinterpret_cast<u32x4*>(dst + o) = val;
      }
      __builtin_amdgcn_s_waitcnt(0xc07f);
      __builtin_amdgcn_wave_barrier();
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < RB; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      bool ok;
      OutT* dst = row_ptr(i * 32 + 8 * (r >> 2) + 4 * lh + (r & 3), ok);
#pragma unroll
      for (int b = 0; b < CB; ++b) {
        const int64_t o = (cb0 + b) * 32 + (lane & 31);
        if (ok && o < p.Cout) Elem<OutT>::store(dst + o * p.ys1, out_val(acc[i][b][r], b));
      }
    }
}

template <int DT, int RB>
void launch_img_rb(const KnnParams& p, const ImgTables& t, int cb, int n_ct, int64_t total, int64_t padded,
                   int vec_out, hipStream_t s) {
  const dim3 grid(static_cast<unsigned>(padded)), block(IM_THREADS);
  if (cb == 2) hipLaunchKernelGGL((knnconv_img_kernel<DT, RB, 2>), grid, block, 0, s, p, t, n_ct, total, padded, vec_out);
  else hipLaunchKernelGGL((knnconv_img_kernel<DT, RB, 1>), grid, block, 0, s, p, t, n_ct, total, padded, vec_out);
}

template <int DT>
void launch_img_dt(const KnnParams& p, const ImgTables& t, int rb, int cb, int n_ct, int64_t total, int64_t padded,
                   int vec_out, hipStream_t s) {
  if (rb == 4) launch_img_rb<DT, 4>(p, t, cb, n_ct, total, padded, vec_out, s);
  else if (rb == 2) launch_img_rb<DT, 2>(p, t, cb, n_ct, total, padded, vec_out, s);
  else launch_img_rb<DT, 1>(p, t, cb, n_ct, total, padded, vec_out, s);
}

// Weight in this kernel's fragment order: 1 KB fragments f = (it * ncb + cb) * 2 + h with
// it = chunk * n_ref + p and slot v = order[p] (v = p without an order); lane l of fragment f
// holds w[o = cb * 32 + l % 32][c * n_ref + v] (zero for o >= c_out or c >= c_in), chunk-relative
// channel 16 h + 8 (l / 32) + e (bf16, e < 8), 8 h + 4 (l / 32) + e (fp32, e < 4),
// 32 (l / 32) + 16 h + e (e4m3, divided by w_scale[o], e < 16).
__global__ void pack_weight_img_kernel(const float* w_ref, int64_t c_out, int64_t c_in, int64_t n_ref, void* out,
                                       int dtype, int64_t ncb, int64_t total, const int32_t* order,
                                       const float* w_scale, int32_t* flag) {
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (idx >= total) return;
  const int eb = dtype == FOVI_F8E4M3 ? 4 : (dtype == FOVI_BF16 ? 3 : 2);
  const int e = static_cast<int>(idx & ((1 << eb) - 1));
  const int l = static_cast<int>((idx >> eb) & 63);
  const int64_t frag = idx >> (eb + 6);
  const int h = static_cast<int>(frag & 1);
  const int64_t cb = (frag >> 1) % ncb;
  const int64_t it = (frag >> 1) / ncb;
  const int64_t pos = it % n_ref, cc = it / n_ref;
  const int64_t v = order ? order[pos] : pos;
  const int64_t o = cb * 32 + (l & 31);
  const int lh = l >> 5;
  const int64_t c = dtype == FOVI_F8E4M3 ? cc * 64 + lh * 32 + h * 16 + e
                                         : (dtype == FOVI_BF16 ? cc * 32 + h * 16 + lh * 8 + e
                                                               : cc * 16 + h * 8 + lh * 4 + e);
  const bool in = o < c_out && c < c_in;
  const float val = in ? w_ref[o * c_in * n_ref + c * n_ref + v] : 0.0f;
  bool bad;
  if (dtype == FOVI_F8E4M3) {
    const uint8_t q = in ? f32_to_e4m3(val / w_scale[o]) : 0;
    static_cast<uint8_t*>(out)[idx] = q;
    bad = (q & 0x7fu) == 0x7fu;
  } else if (dtype == FOVI_BF16) {
    const uint16_t q = f32_to_bf16_bits(val);
    static_cast<uint16_t*>(out)[idx] = q;
    bad = (q & 0x7f80u) == 0x7f80u;
  } else {
    static_cast<float*>(out)[idx] = val;
    bad = (__float_as_uint(val) & 0x7f800000u) == 0x7f800000u;
  }
  if (bad) *flag = 1;   // every writer stores the same value
}

int64_t img_chunk(int dtype) { return dtype == FOVI_F8E4M3 ? 64 : (dtype == FOVI_BF16 ? 32 : 16); }
int64_t img_blocks(int64_t c_out) { return (c_out + 63) / 64 * 2; }

}  // namespace

// 1: launched, 0: the arguments do not fit this kernel (nothing launched).
int launch_knnconv_img(const KnnParams& p, const fovi_knnconv_args* a, hipStream_t s) {
  if (!a->img_ent || !a->img_points || !a->img_nact || !a->img_flag) return 0;
  const int dt = a->x_dtype;
  if (a->w_dtype != dt || p.w_c_slot != p.C) return 0;
  const int es = dt == FOVI_F32 ? 4 : (dt == FOVI_BF16 ? 2 : (dt == FOVI_F8E4M3 ? 1 : 0));
  if (es == 0 || a->y_dtype != (dt == FOVI_F32 ? FOVI_F32 : FOVI_BF16) || (dt == FOVI_F8E4M3 && !p.w_scale)) return 0;
  const int64_t al = 16 / es;
  if (p.xs1 != 1 || p.xs0 < 0 || p.xs2 < 0 || p.xs0 % al != 0 || p.xs2 % al != 0 || p.C % al != 0 ||
      (reinterpret_cast<uintptr_t>(p.x) | reinterpret_cast<uintptr_t>(p.w) | reinterpret_cast<uintptr_t>(a->img_ent)) %
              16 != 0)
    return 0;
  const int ib = a->img_ib, pp = a->img_pp, rows = ib * pp;
  if (ib < 16 || ib > 128 || (ib & (ib - 1)) != 0 || (rows != 32 && rows != 64 && rows != 128)) return 0;
  if (a->img_groups <= 0 || a->img_groups * pp < p.Nout) return 0;
  // 32-bit buffer offsets below IM_NONE
  const int64_t imgs = p.B < ib ? p.B : ib;
  const int64_t lim = (int64_t(1) << 31) - 256;
  if (p.xs0 * es >= lim || p.xs2 * es >= lim || p.Nin >= lim ||
      (p.xs0 > 0 && (imgs - 1) > lim / (p.xs0 * es)) || (p.xs2 > 0 && (p.Nin - 1) > lim / (p.xs2 * es)) ||
      (imgs - 1) * p.xs0 * es + (p.Nin - 1) * p.xs2 * es + p.C * es >= lim)
    return 0;
  const int cb = a->img_cb == 2 ? 2 : 1;
  ImgTables t;
  t.ent = reinterpret_cast<const u32x4*>(a->img_ent);
  t.points = a->img_points; t.nact = a->img_nact; t.flag = a->img_flag;
  t.groups = a->img_groups; t.pp = pp; t.ib = ib;
  t.ibs = __builtin_ctz(static_cast<unsigned>(ib));
  t.ncb = static_cast<int>(img_blocks(p.Cout));
  const int64_t n_ct = (p.Cout + cb * 32 * IM_WAVES - 1) / (cb * 32 * IM_WAVES);
  const int64_t total = n_ct * t.groups * ((p.B + ib - 1) / ib);
  const int64_t padded = (total + 7) / 8 * 8;
  if (padded > 0x7fffffff || p.V * t.ncb > 0x7fffffff / 64) return 0;
  const int64_t op = dt == FOVI_F32 ? 4 : 8;
  const int vec_out = p.ys1 == 1 && p.ys2 % op == 0 && p.ys0 % op == 0 && p.Cout % op == 0 &&
                      reinterpret_cast<uintptr_t>(p.y) % 16 == 0;
  const int rb = rows / 32;
  if (dt == FOVI_BF16) launch_img_dt<FOVI_BF16>(p, t, rb, cb, static_cast<int>(n_ct), total, padded, vec_out, s);
  else if (dt == FOVI_F32) launch_img_dt<FOVI_F32>(p, t, rb, cb, static_cast<int>(n_ct), total, padded, vec_out, s);
  else launch_img_dt<FOVI_F8E4M3>(p, t, rb, cb, static_cast<int>(n_ct), total, padded, vec_out, s);
  return 1;
}

}  // namespace fovi

extern "C" int64_t fovi_knnconv_weight_img_elems(int64_t c_out, int64_t c_in, int64_t n_ref, int32_t dtype) {
  using namespace fovi;
  if (c_out <= 0 || c_in <= 0 || n_ref <= 0 || dtype < FOVI_F32 || dtype > FOVI_F8E4M3) return -1;
  const int64_t ch = img_chunk(dtype);
  return (c_in + ch - 1) / ch * ch * n_ref * img_blocks(c_out) * 32;
}

extern "C" int fovi_knnconv_pack_weight_img(const float* w_ref, int64_t c_out, int64_t c_in, int64_t n_ref, void* w_frag,
                                            int32_t dtype, const int32_t* slot_order, const float* w_scale,
                                            int32_t* flag, void* stream) {
  using namespace fovi;
  clear_error();
  if (!w_ref || !w_frag || !flag) { set_error("fovi_knnconv_pack_weight_img: null pointer"); return 1; }
  const int64_t total = fovi_knnconv_weight_img_elems(c_out, c_in, n_ref, dtype);
  if (total < 0 || (dtype == FOVI_F8E4M3 && !w_scale)) {
    set_error("fovi_knnconv_pack_weight_img: bad sizes, dtype %d, or e4m3 without w_scale", dtype);
    return 1;
  }
  const int64_t blocks = (total + 255) / 256;
  if (blocks > 0x7fffffff) { set_error("fovi_knnconv_pack_weight_img: weight too large"); return 1; }
  hipLaunchKernelGGL(pack_weight_img_kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), w_ref, c_out, c_in, n_ref, w_frag, dtype, img_blocks(c_out),
                     total, slot_order, w_scale, flag);
  return check_launch("fovi_knnconv_pack_weight_img");
}

// Host: groups of `pp` output points with similar slot sets. Within each window of `window`
// consecutive points (of point_order, or of the index order) a group starts at the unassigned point
// with most slots and takes, one at a time, the point that adds fewest slots to the union (ties: most
// slots shared, then the lowest index). With ent == NULL only the groups' union sizes are counted, over every `stride`-th window.
namespace fovi {
namespace {

struct ImgTableArgs {
  const int32_t *slot_ptr, *nbr;
  int64_t n_out, k, n_ref;
  const int32_t *slot_order, *point_order;
  int64_t pp, window, stride;
  uint32_t* ent;
  int32_t *points, *nact;
};

// The groups of windows [q0, q1) (window q starts at point q * window * stride); every window but
// the last has ceil(window / pp) groups, so each knows where its own begin. Returns the sum of the
// groups' union sizes.
int64_t img_table_windows(const ImgTableArgs& a, int64_t q0, int64_t q1) {
  const int64_t n_ref = a.n_ref, pp = a.pp, words = (n_ref + 63) / 64, per_window = (a.window + pp - 1) / pp;
  auto point = [&](int64_t i) -> int64_t { return a.point_order ? a.point_order[i] : i; };
  // in registers: the host baseline's popcount builtin is a library call
  auto pop = [](uint64_t b) -> int32_t {
    b -= (b >> 1) & 0x5555555555555555ull;
    b = (b & 0x3333333333333333ull) + ((b >> 2) & 0x3333333333333333ull);
    return static_cast<int32_t>((((b + (b >> 4)) & 0x0f0f0f0f0f0f0f0full) * 0x0101010101010101ull) >> 56);
  };
  const int64_t most = a.n_out < a.window ? a.n_out : a.window;
  std::vector<uint64_t> bits(static_cast<size_t>(most * words)), uni(static_cast<size_t>(words));
  std::vector<int32_t> used_n(static_cast<size_t>(most));
  std::vector<int64_t> group(static_cast<size_t>(pp)), left;
  int64_t sum = 0;
  for (int64_t q = q0; q < q1; ++q) {
    const int64_t w0 = q * a.window * a.stride;
    const int64_t wn = a.n_out - w0 < a.window ? a.n_out - w0 : a.window;
    int64_t groups = q * per_window;
    std::fill(bits.begin(), bits.end(), 0);
    for (int64_t i = 0; i < wn; ++i) {
      const int32_t* sp = a.slot_ptr + point(w0 + i) * n_ref;
      for (int64_t v = 0; v < n_ref; ++v)
        bits[i * words + (v >> 6)] |= static_cast<uint64_t>((sp[v] & 0xffff) != 0) << (v & 63);
      used_n[i] = 0;
      for (int64_t w = 0; w < words; ++w) used_n[i] += pop(bits[i * words + w]);
    }
    left.clear();
    for (int64_t i = 0; i < wn; ++i) left.push_back(i);
    size_t head = 0;                               // pp = 1 takes the points in order
    while (head < left.size()) {
      int64_t n = 0;
      std::fill(uni.begin(), uni.end(), 0);
      while (n < pp && head < left.size()) {
        size_t best = head;
        if (pp > 1) {
          int64_t bs = INT64_MIN;
          for (size_t c = 0; c < left.size(); ++c) {
            int64_t add = used_n[left[c]];
            if (n > 0) {
              add = 0;
              for (int64_t w = 0; w < words; ++w) add += pop(bits[left[c] * words + w] & ~uni[w]);
            }
            const int64_t score = n == 0 ? add : used_n[left[c]] - add - add * 65536;   // shared, then added
            if (score > bs) { bs = score; best = c; }
          }
        }
        const int64_t i = left[best];
        if (pp > 1) left.erase(left.begin() + static_cast<int64_t>(best));
        else ++head;
        for (int64_t w = 0; w < words; ++w) uni[w] |= bits[i * words + w];
        group[n++] = i;
      }
      int64_t na = 0;
      for (int64_t w = 0; w < words; ++w) na += pop(uni[w]);
      sum += na;
      if (a.ent) {
        for (int64_t j = 0; j < pp; ++j)
          a.points[groups * pp + j] = j < n ? static_cast<int32_t>(point(w0 + group[j])) : -1;
        a.nact[groups] = static_cast<int32_t>(na);
        int64_t row = 0;
        for (int pass = 0; pass < 2; ++pass)          // the union's slots in visit order, then the others
          for (int64_t pos = 0; pos < n_ref; ++pos) {
            const int64_t v = a.slot_order ? a.slot_order[pos] : pos;
            const bool used = (uni[v >> 6] >> (v & 63)) & 1;
            if (used != (pass == 0)) continue;
            for (int64_t j = 0; j < pp; ++j) {
              uint32_t* e = a.ent + ((groups * n_ref + row) * pp + j) * 4;
              const int64_t n_j = j < n ? point(w0 + group[j]) : 0;
              const uint32_t sp = j < n ? static_cast<uint32_t>(a.slot_ptr[n_j * n_ref + v]) : 0u;
              const uint32_t cnt = sp & 0xffffu, begin = sp >> 16;
              const int32_t* list = cnt ? a.nbr + n_j * a.k + begin : nullptr;
              e[0] = cnt > 0 ? static_cast<uint32_t>(list[0]) : IM_NONE;
              e[1] = cnt > 1 ? static_cast<uint32_t>(list[1]) : IM_NONE;
              e[2] = cnt << 16 | begin;
              e[3] = static_cast<uint32_t>(pos);
            }
            ++row;
          }
      }
      ++groups;
    }
  }
  return sum;
}

}  // namespace
}  // namespace fovi

// The windows are shared out to up to eight host threads (16384 points, V = 25, pp = 1 / 8, an eight-core
// host: 4.5 / 9.6 ms on one thread, 1.2 / 2.7 ms on eight; 1379 points, V = 9: 0.3 to 0.5 ms).
extern "C" int64_t fovi_knnconv_img_tables(const int32_t* slot_ptr, const int32_t* nbr, int64_t n_out, int64_t k,
                                           int64_t n_ref, const int32_t* slot_order, const int32_t* point_order,
                                           int32_t pp, int64_t window, int64_t stride, uint32_t* ent,
                                           int32_t* points, int32_t* nact, double* mean_union) {
  using namespace fovi;
  clear_error();
  if (!slot_ptr || (!nbr && ent) || n_out <= 0 || k <= 0 || k > 32767 || n_ref <= 0 || pp <= 0 || window <= 0 ||
      stride <= 0 || (ent && (!points || !nact || stride != 1))) {
    set_error("fovi_knnconv_img_tables: bad arguments");
    return -1;
  }
  if (point_order)
    for (int64_t i = 0; i < n_out; ++i)
      if (point_order[i] < 0 || point_order[i] >= n_out) {
        set_error("fovi_knnconv_img_tables: point_order must hold output points");
        return -1;
      }
  if (window > n_out) window = n_out;
  if (stride > n_out) stride = n_out;
  const int64_t step = window * stride, windows = (n_out + step - 1) / step;
  const int64_t left = n_out - (windows - 1) * step, last = left < window ? left : window;
  const int64_t groups = (windows - 1) * ((window + pp - 1) / pp) + (last + pp - 1) / pp;
  const ImgTableArgs a{slot_ptr, nbr, n_out, k, n_ref, slot_order, point_order, pp, window, stride, ent, points, nact};
  int64_t sum = 0;
  bool ok = true;
  try {
    const int64_t cpus = std::thread::hardware_concurrency(), most = cpus < 8 ? cpus : 8;
    const int64_t nt = std::max<int64_t>(1, std::min(most, windows));
    std::vector<int64_t> sums(static_cast<size_t>(nt), -1);
    const auto run = [&](int64_t t) {
      try { sums[t] = img_table_windows(a, windows * t / nt, windows * (t + 1) / nt); } catch (...) {}
    };
    std::vector<std::thread> pool;
    pool.reserve(static_cast<size_t>(nt));
    for (int64_t t = 1; t < nt; ++t) {
      try { pool.emplace_back(run, t); } catch (...) { run(t); }
    }
    run(0);
    for (std::thread& th : pool) th.join();
    for (int64_t s : sums) { ok = ok && s >= 0; sum += s; }
  } catch (...) { ok = false; }
  if (!ok) {
    set_error("fovi_knnconv_img_tables: out of memory");
    return -1;
  }
  if (mean_union) *mean_union = static_cast<double>(sum) / static_cast<double>(groups);
  return groups;
}
