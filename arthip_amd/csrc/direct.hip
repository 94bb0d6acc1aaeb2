// Direct 3x3 convs on the matrix cores for narrow layers (padded NHWC fp16 in
// and out): the head of a model with two to four input channels
// (conv3x3_head).

#include <hip/hip_runtime.h>

#include <cstdint>

#include "conv_args.h"
#include "launch.h"
#include "pack.h"
#include "wino_dev.h"

namespace arthip {

constexpr uint32_t kOob = 0x80000000u;

// ---------------------------------------------------------------------------
// Head conv, C = 2, 3 or 4 input channels, M = 16 * NB
// ---------------------------------------------------------------------------
//
// In NHWC the three pixels of a kernel row are 3 C contiguous values, so one
// v_mfma_f32_16x16x32_f16 takes the first eight values of all three rows: lane
// (q, j) supplies row q of pixel j (q = 3: zeros). Values 8 .. 11 (C = 3, 4) go
// to a second one laid out the same way (a K = 16 product would hold them, but
// v_mfma_f32_16x16x16_f16 accumulating onto a K = 32 result gave wrong values in
// the result's first two registers). A holds the taps in the same slots (packed
// by winograd_pack, zero where no tap is), its channels permuted so that lane
// (q, j) ends with the contiguous channels 4 NB q .. 4 NB q + 4 NB - 1 of pixel j.
//
// Rows of the padded input start on 4 bytes (Wp is even), pixels of an odd C
// do not: a lane loads the dwords that cover its values and shifts by the
// parity of its pixel. Lanes of q = 3, and pixels past the input, read zeros
// (out-of-range offsets); pixels past the right edge are computed from
// whatever follows their row and never stored.
//
// The write stream bounds it. 3 -> 64 at 1280x720 (123 MB, 118 of them
// written): 172 us in winograd_conv (C padded to 32, element loads, 8-byte
// stores of partial lines), 28 us here (4.4 TB/s). Staging, stores and batches of
// four items as in direct_conv_c1_mfma: one wave's 16 pixels go through its own
// LDS region so that every store instruction covers whole lines, and a batch's
// loads all go out before its first item runs.
template <int C, int NB, int ACT>
__global__ void __launch_bounds__(256) conv3x3_head(DirectRowArgs a) {
  static_assert(C >= 2 && C <= 4, "at most two K = 32 products");
  constexpr int M = 16 * NB;
  constexpr int SEG = 64;
  constexpr int CH = 2 * NB;    // 16-byte chunks per pixel
  constexpr int WCH = 16 * CH;  // chunks of a wave's 16-pixel block
  constexpr int ND = C == 2 ? 3 : (C == 3 ? 5 : 6);  // dwords covering 3 C values
  extern __shared__ __attribute__((aligned(16))) h8 hstage[];
  const int tid = threadIdx.x;
  const int wave = tid >> 6;
  const int lane = tid & 63;
  const int j = lane & 15;  // pixel of the wave's 16 (B column, D column)
  const int q = lane >> 4;  // kernel row (B / A slots), channel quarter of D
  h8* const wl = hstage + wave * WCH;
  auto swz = [](int g) { return g ^ ((g >> 3) & 7); };
  const int rl = lane ^ (((lane >> 4) & 1) << 3);  // chunk of the lane in a store

  h8 wa[NB];
  h8 wb[NB];
  f4 bias4[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const h8* wp = reinterpret_cast<const h8*>(a.w) + (b * 64 + lane) * 2;
    wa[b] = wp[0];
    wb[b] = wp[1];
    bias4[b] = *reinterpret_cast<const f4*>(a.bias + q * 4 * NB + 4 * b);
  }

  const int G = gridDim.x;
  const int slot = (blockIdx.x & 7) * (G >> 3) + (blockIdx.x >> 3);
  const int begin = (int)((int64_t)a.n_items * slot / G);
  const int end = (int)((int64_t)a.n_items * (slot + 1) / G);
  if (begin >= end) return;

  // Item = (n * n_seg + segment) * H + output row.
  auto decode = [&](int item, int& n, int& sg, int& y) {
    const uint32_t t = fdiv((uint32_t)item, a.fd_H);
    y = item - (int)(t * (uint32_t)a.H);
    const uint32_t nn = fdiv(t, a.fd_seg);
    sg = (int)(t - nn * (uint32_t)a.n_seg);
    n = (int)nn;
  };
  const uint32_t img = (uint32_t)a.Hp * (uint32_t)a.Wp * (2 * C);
  // The dwords of padded row y + q, columns x .. x + 2 of this lane's pixel x.
  auto load_b = [&](int item, uint32_t (&d)[ND]) {
    int n, sg, y;
    decode(item, n, sg, y);
    const int x = SEG * sg + 16 * wave + j;
    const char* base = reinterpret_cast<const char*>(a.in) + (int64_t)n * img;
    const __amdgpu_buffer_rsrc_t rs =
        __builtin_amdgcn_make_buffer_rsrc((void*)base, (short)0, (int)img, 0x00020000);
    const uint32_t o =
        q < 3 ? ((uint32_t)((y + q) * a.Wp + x) * (2 * C)) & ~3u : kOob;
    if constexpr (C == 2) {
      const auto v = __builtin_amdgcn_raw_buffer_load_b96(rs, o, 0, 0);
#pragma unroll
      for (int i = 0; i < 3; ++i) d[i] = v[i];
    } else {
      const u4 v = __builtin_amdgcn_raw_buffer_load_b128(rs, o, 0, 0);
#pragma unroll
      for (int i = 0; i < 4; ++i) d[i] = v[i];
      if constexpr (C == 3) {
        d[4] = __builtin_amdgcn_raw_buffer_load_b32(rs, o + 16, 0, 0);
      } else {
        const u2 t = __builtin_amdgcn_raw_buffer_load_b64(rs, o + 16, 0, 0);
        d[4] = t[0];
        d[5] = t[1];
      }
    }
  };

  const uint32_t sh = (C & 1) != 0 ? (uint32_t)(j & 1) * 16 : 0;  // SEG and 16 are even
  constexpr int kBatch = 4;
  auto item = [&](int it, const uint32_t (&d)[ND]) {
    int n, sg, y;
    decode(it, n, sg, y);
    const int x0 = SEG * sg;
    u4 lo;
    u4 hi = {0, 0, 0, 0};
    if constexpr (C == 2) {
      lo = u4{d[0], d[1], d[2], 0};
    } else if constexpr (C == 3) {
#pragma unroll
      for (int i = 0; i < 4; ++i) lo[i] = __builtin_amdgcn_alignbit(d[i + 1], d[i], sh);
      hi[0] = (d[4] >> sh) & 0xffffu;
    } else {
      lo = u4{d[0], d[1], d[2], d[3]};
      hi = u4{d[4], d[5], 0, 0};
    }
    const h8 bl = __builtin_bit_cast(h8, lo);
    const h8 bh = __builtin_bit_cast(h8, hi);
    char* ob = reinterpret_cast<char*>(a.out) + (((int64_t)n * a.Hp + y + 1) * a.Wp + x0 + 1) * M * 2;
    const int valid = min(SEG, a.W - x0);
    const __amdgpu_buffer_rsrc_t rs =
        __builtin_amdgcn_make_buffer_rsrc((void*)ob, (short)0, valid * M * 2, 0x00020000);
    auto prod = [&](int b) {
      f4 d0 = bias4[b];
      d0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(wa[b], bl, d0, 0, 0, 0);
      if constexpr (C > 2) d0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(wb[b], bh, d0, 0, 0, 0);
      return strip_act4<ACT>(d0);
    };
#pragma unroll
    for (int m = 0; m < NB / 2; ++m) {
      const h4 v0 = prod(2 * m), v1 = prod(2 * m + 1);
      wl[swz(j * CH + q * (NB / 2) + m)] = __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7);
    }
    // The wave's block is bytes [16 * wave * M * 2, + 16 * M * 2) of the row
    // segment; pixels past the image's right edge fall outside the resource.
    const uint32_t wbase = (uint32_t)(16 * wave * M * 2);
#pragma unroll
    for (int st = 0; st < WCH / 64; ++st) {
      const int g = 64 * st + rl;
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4, wl[swz(g)]), rs, wbase + 16 * g, 0, 0);
    }
  };
  for (int it = begin; it < end; it += kBatch) {
    uint32_t v[kBatch][ND];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) load_b(min(it + u, end - 1), v[u]);
#pragma unroll
    for (int u = 0; u < kBatch; ++u)
      if (it + u < end) item(it + u, v[u]);
  }
}

// ---------------------------------------------------------------------------
// Host launchers
// ---------------------------------------------------------------------------

namespace {

using RowKernel = void (*)(DirectRowArgs);

template <int C, int NB>
RowKernel head_kernel_act(int act) {
  return act == kActRelu   ? conv3x3_head<C, NB, kActRelu>
         : act == kActSilu ? conv3x3_head<C, NB, kActSilu>
                           : conv3x3_head<C, NB, kActNone>;
}

template <int C>
RowKernel head_kernel(int M, int act) {
  return M == 32 ? head_kernel_act<C, 2>(act) : M == 64 ? head_kernel_act<C, 4>(act)
                                                        : head_kernel_act<C, 6>(act);
}

bool aligned16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

// Padded fp16 image and work items within the kernels' 32-bit offsets.
bool fits32(int64_t N, int64_t H, int64_t W, int64_t ch, int64_t seg) {
  const int64_t lim = (int64_t)1 << 31;
  return padded_rows(H) * padded_cols(W) * ch * 2 < lim && N * ((W + seg - 1) / seg) * H < lim;
}

DirectRowArgs row_args(const WinoArgs& w, int seg) {
  DirectRowArgs a{};
  a.in = w.in;
  a.bias = w.epi.bias;
  a.skip0 = w.epi.skip0 ? w.epi.skip0 : w.epi.skip1;
  a.skip1 = w.epi.skip0 ? w.epi.skip1 : nullptr;
  a.out = reinterpret_cast<uint16_t*>(w.epi.out);
  a.w = w.u + direct_rows_offset(w.C, w.M);
  a.N = w.N;
  a.H = w.H;
  a.W = w.W;
  a.M = w.M;
  a.act = w.epi.act;
  a.Hp = (int32_t)padded_rows(w.H);
  a.Wp = (int32_t)padded_cols(w.W);
  a.n_seg = (w.W + seg - 1) / seg;
  a.n_items = (int32_t)((int64_t)w.N * a.n_seg * w.H);
  a.fd_H = make_fastdiv((uint32_t)w.H);
  a.fd_seg = make_fastdiv((uint32_t)a.n_seg);
  return a;
}

hipError_t launch_rows_kernel(RowKernel fn, const DirectRowArgs& a, int threads, size_t lds,
                              hipStream_t s) {
  if (lds > 65536) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
  }
  int occ = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, reinterpret_cast<const void*>(fn), threads,
                                                   lds) != hipSuccess ||
      occ < 1)
    occ = 1;
  int64_t grid = (int64_t)cu_count() * occ;
  if (grid > a.n_items) grid = a.n_items;
  grid = (grid + 7) / 8 * 8;
  hipLaunchKernelGGL(fn, dim3((unsigned)grid), dim3(threads), lds, s, a);
  return hipGetLastError();
}

// Padded NHWC fp16 on both sides, no Clip, no DepthToSpace.
bool inner_epilogue(const WinoArgs& w) {
  return !w.in_nchw && w.epi.out_kind == kOutPadded && w.epi.dts_b < 2 && !w.epi.do_clip &&
         (w.epi.act == kActNone || w.epi.act == kActRelu || w.epi.act == kActSilu);
}

}  // namespace

// The head kernel needs dword-aligned input rows and 16-byte stores; a
// residual input on such a conv stays on winograd_conv.
bool conv_head_eligible(const WinoArgs& w) {
  return inner_epilogue(w) && direct_head_shape(w.C, w.M) && w.epi.skip0 == nullptr &&
         w.epi.skip1 == nullptr && aligned16(w.in) && aligned16(w.epi.out) &&
         fits32(w.N, w.H, w.W, w.C, 64);
}

hipError_t launch_conv_head(const WinoArgs& w, hipStream_t s) {
  if (!conv_head_eligible(w)) return hipErrorInvalidValue;
  const DirectRowArgs a = row_args(w, 64);
  const RowKernel fn = w.C == 2   ? head_kernel<2>(w.M, a.act)
                       : w.C == 3 ? head_kernel<3>(w.M, a.act)
                                  : head_kernel<4>(w.M, a.act);
  return launch_rows_kernel(fn, a, 256, (size_t)4 * 16 * w.M * 2, s);
}

}  // namespace arthip
