// Weight gradient of the kNN convolution for gfx950, without the slot-sum matrix.
//
// dW[o, c * V + v] = sum over images b and over the (output n, input i) pairs whose
// neighbour i sits in slot v of n of dy[b, n, o] * x[b, i, c]: for every slot a GEMM whose
// reduction runs over that slot's pair list (the sum of a collision slot is linear, so its
// pairs enter one by one). The pairs come in segments (one slot, one chunk of output
// points); a workgroup owns one segment, a group of images and one TO x TC (o, c) tile: 256
// channels, or 128 where the layer has no more (96 x 256 channels on a 256 x 256 tile spend
// 62% of the products on zeros). Its waves hold 128 x 64 fp32 blocks (8 blocks of
// v_mfma_f32_32x32x16_bf16): eight of them, two per SIMD so one wave's memory waits overlap
// the other's MFMAs, or two workgroups of four (or four of two) per CU. Workgroups are
// numbered slot-fastest and mapped XCD by XCD, so the V workgroups of a chunk share one L2.
//
// Per step of K = 64 pairs (32 with the smaller tiles) the workgroup loads the dy rows and the x
// rows (16-byte chunks, a full row per 32 or 16 lanes) into LDS in their natural [pair][channel]
// layout, double buffered one step ahead. Both MFMA operands need the pair index contiguous per
// lane, which the transposed LDS read ds_read_b64_tr_b16 delivers: within a 16-lane group, lane j
// addresses four channels of pair row k0 + j/4 and lane i receives channel i of pairs k0 ..
// k0 + 3. Rows are 576 (320) bytes apart so those reads hit 64 distinct banks. Per-workgroup partial
// tiles go to a caller workspace; a second kernel sums them into the reference weight layout
// (column c * V + v), fp32.
#include "common.h"

namespace fovi {
namespace {

// Tile of the output (O) or input (C) channels: 256, or 128 for up to 128 channels.
inline int64_t dw_tile(int64_t channels) { return channels <= 128 ? 128 : 256; }

template <int TO, int TC> struct DwTile {
  static constexpr int NT = (TO / 128) * (TC / 64) * 64;       // threads: a wave per 128 x 64 block
  static constexpr int K = TO == 256 && TC == 256 ? 64 : 32;   // pairs per step
  static constexpr int GO = TO / 8, GC = TC / 8;               // 16-byte chunks per row
  static constexpr int RO = K * GO / NT, RC = K * GC / NT;     // rows per thread and step
  static constexpr int SO = TO * 2 + 64, SC = TC * 2 + 64;     // LDS bytes per row (64 bytes of bank skew)
  static constexpr int BUF = K * (SO + SC);                    // one step
  static constexpr int LDS = 2 * BUF;                          // 256 x 256: 147,456 bytes
};

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4v __attribute__((ext_vector_type(4)));

struct DwParams {
  const uint16_t* x;
  int64_t xs0, xs2;                // x[b * xs0 + i * xs2 + c]
  const uint16_t* dy;
  int64_t ds0, ds2;                // dy[b * ds0 + n * ds2 + o]
  int64_t B, C, Cout, Nin, Nout, V;
  const int32_t* pair_off;         // [NQ * V + 1], segment q * V + v
  const int32_t* pairs;            // (n, i) per pair; n < 0 pads
  int64_t NQ, ipg, S, tiles_o, tiles_c, to, tc;
  float* part;                     // [S, NQ, V, tiles_o, tiles_c, to, tc]
};

__device__ __forceinline__ s16x4 tr_read(const uint8_t* lds_base, int byte_off) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) s16x4*)(reinterpret_cast<uintptr_t>(lds_base) + byte_off));
}

template <int TO, int TC>
__global__ __launch_bounds__((DwTile<TO, TC>::NT), (TO == 256 && TC == 256 ? 1 : 2)) void knnconv_dw_kernel(
    DwParams p, int64_t total, int64_t padded) {
  typedef DwTile<TO, TC> D;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int64_t L = xcd_tile(blockIdx.x, padded);
  if (L >= total) return;                       // whole workgroup: before any barrier
  const int64_t v = L % p.V;
  int64_t rest = L / p.V;
  const int64_t tc = rest % p.tiles_c;
  rest /= p.tiles_c;
  const int64_t to = rest % p.tiles_o;
  rest /= p.tiles_o;
  const int64_t q = rest % p.NQ;
  const int64_t split = rest / p.NQ;
  const int64_t o0 = to * TO, c0 = tc * TC;

  // wave (wm, wn) holds o rows wm*128 .. +127, c columns wn*64 .. +63
  constexpr int WN = TC / 64;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, wm = wave / WN, wn = wave % WN;
  const int64_t seg = q * p.V + v;
  const int64_t P0 = p.pair_off[seg], P1 = p.pair_off[seg + 1];
  const int64_t steps_img = (P1 - P0 + D::K - 1) / D::K;     // the last step's tail reads as pads
  const int64_t b_beg = split * p.ipg;
  const int64_t steps = steps_img * (min(p.B, b_beg + p.ipg) - b_beg);

  // load task: dy rows t/GO + (NT/GO) r, 16-byte chunk t%GO of the row, x rows alike; chunks past
  // the channels load chunk 0 and pads load row 0, both masked to zero when stored
  const int go = t % D::GO, po = t / D::GO, gc = t % D::GC, pc = t / D::GC;
  const bool oko = o0 + 8 * go < p.Cout, okc = c0 + 8 * gc < p.C;
  const int go1 = oko ? go : 0, gc1 = okc ? gc : 0;

  f32x16 acc[4][2];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

  int2 eo[D::RO], ec[D::RC];                    // pair entries of the step being prefetched (square tiles: eo)
  u32x4v rd[D::RO], rx[D::RC];                  // rows of the step in flight
  uint32_t m = 0;                               // their live bits
  auto load_pairs = [&](int64_t st) __attribute__((always_inline)) {
    const int64_t base = P0 + D::K * ((st < steps ? st : 0) % steps_img);
    auto entry = [&](int64_t pi) {
      int2 e = *reinterpret_cast<const int2*>(p.pairs + 2 * (pi < P1 ? pi : P1 - 1));
      if (pi >= P1) e.x = -1;                     // past the segment: a pad
      return e;
    };
#pragma unroll
    for (int r = 0; r < D::RO; ++r) eo[r] = entry(base + po + (D::NT / D::GO) * r);
    if constexpr (D::GO != D::GC)
#pragma unroll
      for (int r = 0; r < D::RC; ++r) ec[r] = entry(base + pc + (D::NT / D::GC) * r);
  };
  auto load_rows = [&](int64_t st) __attribute__((always_inline)) {
    const bool on = st < steps;
    const int64_t b = b_beg + (on ? st / steps_img : 0);   // uniform: the image base stays scalar
    const uint16_t* xb = p.x + b * p.xs0 + c0;
    const uint16_t* db = p.dy + b * p.ds0 + o0;
    m = 0;
    // 32-bit element offsets within the image (the host checks they fit)
#pragma unroll
    for (int r = 0; r < D::RO; ++r) {
      const bool live = on && eo[r].x >= 0;
      const uint32_t n = live ? eo[r].x : 0;
      rd[r] = *reinterpret_cast<const u32x4v*>(db + (n * static_cast<uint32_t>(p.ds2) + 8u * go1));
      m |= static_cast<uint32_t>(live && oko) << r;
    }
#pragma unroll
    for (int r = 0; r < D::RC; ++r) {
      const int2 e = D::GO == D::GC ? eo[r] : ec[r];
      const bool live = on && e.x >= 0;
      const uint32_t i = live ? e.y : 0;
      rx[r] = *reinterpret_cast<const u32x4v*>(xb + (i * static_cast<uint32_t>(p.xs2) + 8u * gc1));
      m |= static_cast<uint32_t>(live && okc) << (D::RO + r);
    }
  };
  auto store_rows = [&](int buf) __attribute__((always_inline)) {
    uint8_t* bd = smem + buf * D::BUF;
    uint8_t* bx = bd + D::K * D::SO;
    const u32x4v z = {0, 0, 0, 0};
#pragma unroll
    for (int r = 0; r < D::RO; ++r)
      *reinterpret_cast<u32x4v*>(bd + (po + (D::NT / D::GO) * r) * D::SO + 16 * go) = (m >> r & 1) ? rd[r] : z;
#pragma unroll
    for (int r = 0; r < D::RC; ++r)
      *reinterpret_cast<u32x4v*>(bx + (pc + (D::NT / D::GC) * r) * D::SC + 16 * gc) = (m >> (D::RO + r) & 1) ? rx[r] : z;
  };

  // this lane's transposed-read offsets: 16-lane group G supplies pair rows kb*16 + 8*(G>>1)
  // + li/4 (+4 for the second half) and channels 16*(G&1) + 4*(li%4) of each 32-block
  const int G = lane >> 4, li = lane & 15;
  const int lrow = (G >> 1) * 8 + (li >> 2), lcol = ((G & 1) * 16 + 4 * (li & 3)) * 2;
  const int off_d = lrow * D::SO + lcol + wm * 256, off_x = lrow * D::SC + lcol + wn * 128;

  if (steps > 0) {
    // prologue: step 0 into LDS buffer 0, step 1 in flight, pair entries of step 2 loading
    load_pairs(0);
    load_rows(0);
    store_rows(0);
    load_pairs(1);
    load_rows(1);
    load_pairs(2);
    __syncthreads();
    for (int64_t st = 0; st < steps; ++st) {
      const uint8_t* bd = smem + (st & 1) * D::BUF;
      const uint8_t* bx = bd + D::K * D::SO;
#pragma unroll
      for (int kb = 0; kb < D::K / 16; ++kb) {
        bf16x8 af[4], bf[2];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int off = off_d + kb * 16 * D::SO + i * 64;
          const s16x4 lo = tr_read(bd, off), hi = tr_read(bd, off + 4 * D::SO);
          af[i] = __builtin_bit_cast(bf16x8, s16x8(__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7)));
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const int off = off_x + kb * 16 * D::SC + j * 64;
          const s16x4 lo = tr_read(bx, off), hi = tr_read(bx, off + 4 * D::SC);
          bf[j] = __builtin_bit_cast(bf16x8, s16x8(__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7)));
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[i], bf[j], acc[i][j], 0, 0, 0);
      }
      if (st + 1 < steps) store_rows((st + 1) & 1);  // buffer last read in step st - 1
      load_rows(st + 2);
      load_pairs(st + 3);
      __syncthreads();
    }
  }

  float* out = p.part + (((split * p.NQ * p.V + seg) * p.tiles_o + to) * p.tiles_c + tc) * (TO * TC);
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int o = wm * 128 + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
        const int c = wn * 64 + j * 32 + (lane & 31);
        if (o0 + o < p.Cout && c0 + c < p.C) out[o * TC + c] = acc[i][j][r];   // the reduction reads no others
      }
}

template <int TO, int TC>
int launch_dw(const DwParams& p, int64_t total, int64_t padded, hipStream_t s) {
  if (reserve_dynamic_lds(reinterpret_cast<const void*>(&knnconv_dw_kernel<TO, TC>), DwTile<TO, TC>::LDS) != hipSuccess) {
    set_error("fovi_knnconv_dw: cannot reserve %d bytes of LDS", DwTile<TO, TC>::LDS);
    return 1;
  }
  hipLaunchKernelGGL((knnconv_dw_kernel<TO, TC>), dim3(static_cast<unsigned>(padded)), dim3(DwTile<TO, TC>::NT),
                     (DwTile<TO, TC>::LDS), s, p, total, padded);
  return check_launch("fovi_knnconv_dw");
}

// dW[o, c * V + v] = sum over the (image group, chunk) partial tiles (fp32, in that order; four
// loads in flight per trip). A block takes one o and cc channels: a thread reads along c (the
// partials' fast axis), the sums go through LDS and leave as runs of cc * V consecutive floats
// (written straight from the reading order, one float per 4 V bytes, every line of dW is
// touched V times). Blocks along y take vt slots each; more than one of them only with cc = 1.
__global__ __launch_bounds__(256) void knnconv_dw_reduce_kernel(DwParams p, float* dw, int cc, int ccs, int vt) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  float* out = reinterpret_cast<float*>(smem);                 // [cc][V], V the block's slots
  const int64_t vb = static_cast<int64_t>(blockIdx.y) * vt;
  const int V = static_cast<int>(min(static_cast<int64_t>(vt), p.V - vb));
  const int64_t nc = (p.C + cc - 1) / cc;
  const int64_t o = blockIdx.x / nc, c0 = (blockIdx.x % nc) * cc;
  const int lc = threadIdx.x & (cc - 1), v0 = threadIdx.x >> ccs, dv = 256 >> ccs;
  const int64_t c = c0 + lc;
  const int64_t n = p.S * p.NQ;
  const int64_t stride = p.V * p.tiles_o * p.tiles_c * (p.to * p.tc);   // next (group, chunk)
  if (c < p.C) {
    const int64_t tile = (o / p.to) * p.tiles_c + c / p.tc;
    const float* base = p.part + (vb * p.tiles_o * p.tiles_c + tile) * (p.to * p.tc) + (o % p.to) * p.tc + c % p.tc;
    for (int v = v0; v < V; v += dv) {
      const float* src = base + v * p.tiles_o * p.tiles_c * (p.to * p.tc);
      float sum = 0.0f;
      int64_t sq = 0;
      for (; sq + 4 <= n; sq += 4) {
        float t[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) t[u] = src[(sq + u) * stride];
#pragma unroll
        for (int u = 0; u < 4; ++u) sum += t[u];
      }
      for (; sq < n; ++sq) sum += src[sq * stride];
      out[lc * V + v] = sum;
    }
  }
  __syncthreads();
  const int64_t left = p.C - c0;
  const int count = static_cast<int>(left < cc ? left : cc) * V;
  float* dst = dw + (o * p.C + c0) * p.V + vb;
  for (int i = threadIdx.x; i < count; i += 256) dst[i] = out[i];
}

}  // namespace
}  // namespace fovi

using namespace fovi;

extern "C" int64_t fovi_knnconv_dw_workspace_bytes(int64_t batch, int64_t images_per_group, int64_t n_chunks,
                                                   int64_t c_in, int64_t c_out, int64_t n_ref) {
  if (batch < 1 || images_per_group < 1 || n_chunks < 1 || c_in < 1 || c_out < 1 || n_ref < 1) return -1;
  const int64_t splits = (batch + images_per_group - 1) / images_per_group;
  const int64_t to = dw_tile(c_out), tc = dw_tile(c_in);
  const int64_t tiles = ((c_out + to - 1) / to) * ((c_in + tc - 1) / tc);
  return splits * n_chunks * n_ref * tiles * to * tc * static_cast<int64_t>(sizeof(float));
}

extern "C" int fovi_knnconv_dw(const fovi_knnconv_dw_args* a, void* stream) {
  clear_error();
  if (!a || !a->x || !a->dy || !a->pair_off || !a->pairs || !a->workspace || !a->dw) {
    set_error("fovi_knnconv_dw: null pointer");
    return 1;
  }
  if (a->batch < 1 || a->c_in < 8 || a->c_out < 8 || a->c_in % 8 || a->c_out % 8 || a->n_in < 1 ||
      a->n_out < 1 || a->n_ref < 1 || a->n_chunks < 1 || a->images_per_group < 1 || a->n_in > INT32_MAX ||
      a->n_out > INT32_MAX) {
    set_error("fovi_knnconv_dw: bad sizes (channel counts must be multiples of 8)");
    return 1;
  }
  if (a->n_in * a->x_stride[2] + a->c_in > UINT32_MAX || a->n_out * a->dy_stride[2] + a->c_out > UINT32_MAX) {
    set_error("fovi_knnconv_dw: one image's rows must span fewer than 2^32 elements");
    return 1;
  }
  if (a->x_stride[1] != 1 || a->dy_stride[1] != 1 || a->x_stride[2] % 8 || a->x_stride[0] % 8 ||
      a->dy_stride[2] % 8 || a->dy_stride[0] % 8 || reinterpret_cast<uintptr_t>(a->x) % 16 ||
      reinterpret_cast<uintptr_t>(a->dy) % 16) {
    set_error("fovi_knnconv_dw: x and dy must be channels-last bf16 with 16-byte aligned rows");
    return 1;
  }
  const int64_t need = fovi_knnconv_dw_workspace_bytes(a->batch, a->images_per_group, a->n_chunks, a->c_in,
                                                       a->c_out, a->n_ref);
  if (a->workspace_bytes < need) {
    set_error("fovi_knnconv_dw: workspace %lld bytes, need %lld", (long long)a->workspace_bytes, (long long)need);
    return 1;
  }
  DwParams p;
  p.x = static_cast<const uint16_t*>(a->x); p.xs0 = a->x_stride[0]; p.xs2 = a->x_stride[2];
  p.dy = static_cast<const uint16_t*>(a->dy); p.ds0 = a->dy_stride[0]; p.ds2 = a->dy_stride[2];
  p.B = a->batch; p.C = a->c_in; p.Cout = a->c_out; p.Nin = a->n_in; p.Nout = a->n_out; p.V = a->n_ref;
  p.pair_off = a->pair_off; p.pairs = a->pairs;
  p.NQ = a->n_chunks; p.ipg = a->images_per_group; p.S = (p.B + p.ipg - 1) / p.ipg;
  p.to = dw_tile(p.Cout); p.tc = dw_tile(p.C);
  p.tiles_o = (p.Cout + p.to - 1) / p.to; p.tiles_c = (p.C + p.tc - 1) / p.tc;
  p.part = static_cast<float*>(a->workspace);
  const int64_t total = p.S * p.NQ * p.V * p.tiles_o * p.tiles_c;
  const int64_t padded = (total + 7) / 8 * 8;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int rc = p.to == 256 ? (p.tc == 256 ? launch_dw<256, 256>(p, total, padded, s) : launch_dw<256, 128>(p, total, padded, s))
                             : (p.tc == 256 ? launch_dw<128, 256>(p, total, padded, s) : launch_dw<128, 128>(p, total, padded, s));
  if (rc) return rc;
  // channels per reduction block: 32, fewer where their V sums pass 64 KB of LDS; slots in pieces where
  // one channel's do
  constexpr int64_t sums = 64 * 1024 / 4;
  int ccs = 5;
  while (ccs > 0 && (p.V << ccs) > sums) --ccs;
  const int64_t vt = p.V < sums ? p.V : sums, pieces = (p.V + vt - 1) / vt;
  const int64_t blocks = p.Cout * ((p.C + (1 << ccs) - 1) >> ccs);
  if (blocks > 0x7fffffff || pieces > 65535) {
    set_error("fovi_knnconv_dw: c_out=%lld x c_in=%lld x n_ref=%lld too large", (long long)p.Cout, (long long)p.C,
              (long long)p.V);
    return 1;
  }
  hipLaunchKernelGGL(knnconv_dw_reduce_kernel, dim3(static_cast<unsigned>(blocks), static_cast<unsigned>(pieces)), dim3(256),
                     static_cast<size_t>((vt << ccs) * 4), s, p, a->dw, 1 << ccs, ccs, static_cast<int>(vt));
  return check_launch("fovi_knnconv_dw(reduce)");
}
