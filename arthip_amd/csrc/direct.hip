// Direct 3x3 convs on the matrix cores for narrow layers, padded NHWC fp16 in
// and out: the head of a model with two to four input channels (conv3x3_head)
// and body convs of 16 to 48 channels (conv3x3_rows). For the 32-channel model,
// two convs in one launch at either boundary: the one-channel head and the conv
// after it (conv3x3_head_pair), the last conv and the tail (conv3x3_tail_pair).

#include <hip/hip_runtime.h>

#include <cstdint>

#include "conv_args.h"
#include "launch.h"
#include "pack.h"
#include "plan_rules.h"
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
// to a second one laid out the same way. (A K = 16 product would hold them, but
// hipcc issues a v_mfma_f32_16x16x16_f16 that adds to a K = 32 result right behind
// it, without wait states, as it does for products of one shape; the first two
// registers of the sum were then wrong, as if read before they were written. No
// kernel adds one shape onto another.) A holds the taps in the same slots (packed
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
  const int begin = split_begin(a.split, slot);
  const int end = split_begin(a.split, slot + 1);
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
// Narrow body conv, C = 16 .. 48 (C % 8 == 0), M <= 16 * OB <= 48 (M % 8 == 0)
// ---------------------------------------------------------------------------
//
// In NHWC the three pixels of a kernel row are 3 C contiguous values, so a
// kernel row is KR = ceil(3 C / 32) products of v_mfma_f32_16x16x32_f16: B is 16
// output pixels x 32 values of a row, read from LDS as 16 bytes per lane at the
// pixel's own offset (values past the third pixel are masked to zero), A the
// taps of 16 output channels, held in VGPRs (12 KR OB of them) for the whole
// launch. 9 C products per output are more than Winograd's, but nothing is
// transformed and no V' goes through LDS: the matrix work of these widths is
// below the time of their memory traffic.
//
// One wave per workgroup; it walks down a segment of up to OPX = 30 or 62 output
// pixels, one row per step, on its own: its input rows (two pixels more) come
// by 16-byte buffer -> LDS copies into a private ring of R slots, LA rows ahead
// of the step that reads them, and only the wave's own count of outstanding
// memory instructions orders ring and copies, no barrier. Every step issues the
// same instructions on every path (copies past the run and stores past the
// segment have out-of-range offsets): NSK residual copies, NI row copies, NS
// stores.
//
// Epilogue: bias in the accumulators, one rounding to fp16, activation, then the
// residual inputs in fp16. The channels of A's rows are permuted (pack.h) so
// that a lane holds 4 OB contiguous channels of its pixel; they go to the
// staging slot (with residual inputs the slot that already holds the first
// residual's row, read and overwritten in place) and leave linearly, whole lines
// per store instruction.
//
// LDS banks: a 16-byte read serves lanes 0-3, 12-15, 20-27 of each half wave
// together, then the other 16 (measured: equal units of 16 bytes mod 256 slow a
// read only within these sets). Under that the 32- and 96-byte pixels of
// C = 16 and 48 are conflict-free as they are; C = 32 stores 16-byte group g of
// ring pixel p at g ^ (2 ((p >> 2) & 1)) (on the copies' source side), which is
// too; C = 24 and 40 read two-way.
//
// The stream through memory bounds it at full frames (32 -> 32 with a residual at
// 1080p, 398 MB: 88 us in the strip kernel it ran on before, 63 here, 6.5 TB/s).
// On nine-row runs nothing does alone (48 -> 48 + ReLU at 541x963, 100 MB: 65 us
// in winograd_conv, 30 here; 3.8 TB/s, matrix units 32% busy, LDS 21%): each
// run's first rows and a wave's own chain a step, two waves per SIMD. 32 -> 32 +
// ReLU at 540x960 (66 MB): 24 and 17 us; 16 -> 16 at 1080p (133 MB): 68 and 26.
// (Kernel times; whole calls take about 1 us more.) Its error against 64 bits is a
// third of Winograd's (2.1e-4 against 6.1e-4): no transform rounds its inputs.
//
// C = 24 and 40 take four tiles a step, whose ring rows are whole copies, and two
// where those are the slower form (rows_two_tiles).
template <int C, int OB, int NSKIP, int TILES = C % 16 == 0 ? 2 : 4>
struct RowsL {
  static constexpr int T = TILES;        // 16-pixel tiles per step
  static constexpr int IPX = 16 * T;     // input pixels per ring row
  static constexpr int OPX = IPX - 2;    // output pixels per segment, at most
  static constexpr int PXB = 2 * C;      // input bytes per pixel
  static constexpr int KR = (3 * C + 31) / 32;
  static constexpr int VO = 3 * C / 8 - 4 * (KR - 1);  // octets of the last product
  // Copies per row (C = 24 and 40 with two tiles: half of the last out of range).
  static constexpr int NI = (IPX * PXB + 1023) / 1024;
  static constexpr int SLOT = NI * 1024;
  static constexpr int LA = 2;
  static constexpr int R = LA + 3;
  static constexpr int NS = IPX * 32 * OB / 1024;  // stores per row
  static constexpr int SSLOT = NS * 1024;
  static constexpr int NSK = NSKIP * NS;
  static constexpr int STG = R * SLOT;
  // Reads of the last tile's unused columns run past the last slot.
  static constexpr size_t lds_bytes() { return STG + (NSKIP == 0 ? 1 : 2 * NSKIP) * SSLOT; }
  static_assert((LA - 1) * (NI + NSK) + LA * NS < 64 && 2 * NI + NS + NSK < 64, "vmcnt field");
  static_assert(NS <= (LA + 1) * NI, "the first residual row's wait");
  // Last byte read in a slot: the last pixel's row of KR products.
  static_assert((IPX - 1) * PXB + 64 * KR - SLOT <= SSLOT, "reads stay inside the LDS");
};

// Three input rows (ring slots at row[0..2]) times the taps, onto acc: B of tile t,
// product kc of a row at byte rb[.] + 16 * PXB * t (+ 64 * kc unswizzled).
template <class L, int OB, int NRB>
__device__ __forceinline__ void rows_fold(const h8 (&wa)[3][L::KR][OB], const char* const (&row)[3],
                                          const int (&rb)[NRB], uint32_t vmask, f4 (&acc)[L::T][OB]) {
  constexpr int T = L::T, KR = L::KR;
#pragma unroll
  for (int dy = 0; dy < 3; ++dy)
#pragma unroll
    for (int kc = 0; kc < KR; ++kc) {
      h8 v[T];
#pragma unroll
      for (int t = 0; t < T; ++t) {
        const char* p = row[dy] + (NRB > 1 ? rb[kc % NRB] : rb[0] + 64 * kc) + 16 * L::PXB * t;
        v[t] = *reinterpret_cast<const h8*>(p);
        if (L::VO != 4 && kc == KR - 1)
          v[t] = __builtin_bit_cast(h8, __builtin_bit_cast(u4, v[t]) & u4{vmask, vmask, vmask, vmask});
      }
#pragma unroll
      for (int t = 0; t < T; ++t)
#pragma unroll
        for (int b = 0; b < OB; ++b)
          acc[t][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wa[dy][kc][b], v[t], acc[t][b], 0, 0, 0);
    }
}

// One input row times the taps of the three kernel rows, each onto its own sums
// (acc[dy]): the row's values are read from LDS once. C = 32's swizzled rows.
template <class L, int OB>
__device__ __forceinline__ void rows_fold_once(const h8 (&wa)[3][L::KR][OB], const char* row, const int (&rb)[L::KR],
                                               f4 (&acc)[3][L::T][OB]) {
  constexpr int T = L::T, KR = L::KR;
  static_assert(L::VO == 4, "no masked values");
#pragma unroll
  for (int kc = 0; kc < KR; ++kc) {
    h8 v[T];
#pragma unroll
    for (int t = 0; t < T; ++t) v[t] = *reinterpret_cast<const h8*>(row + rb[kc] + 16 * L::PXB * t);
#pragma unroll
    for (int dy = 2; dy >= 0; --dy)
#pragma unroll
      for (int t = 0; t < T; ++t)
#pragma unroll
        for (int b = 0; b < OB; ++b)
          acc[dy][t][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wa[dy][kc][b], v[t], acc[dy][t][b], 0, 0, 0);
  }
}

// One staged output row leaves linearly: NS whole-kilobyte stores from lin.
template <int NS, int AUX>
__device__ __forceinline__ void rows_store(const char* lin, __amdgpu_buffer_rsrc_t ro, int lane) {
#pragma unroll
  for (int i = 0; i < NS; ++i)
    __builtin_amdgcn_raw_buffer_store_b128(*reinterpret_cast<const u4*>(lin + 1024 * i), ro,
                                           (uint32_t)(1024 * i + 16 * lane), 0, AUX);
}

template <int C, int OB, int NSKIP, int TILES>
__global__ void __launch_bounds__(64)
    __attribute__((amdgpu_waves_per_eu(2)))
conv3x3_rows(DirectRowArgs a) {
  using L = RowsL<C, OB, NSKIP, TILES>;
  constexpr int T = L::T, KR = L::KR, NI = L::NI, NS = L::NS, NSK = L::NSK, LA = L::LA, R = L::R;
  constexpr bool SWZ = C == 32;
  extern __shared__ __attribute__((aligned(16))) char rlds[];
  const int lane = threadIdx.x;
  const int j = lane & 15;
  const int q = lane >> 4;

  const int G = gridDim.x;
  const int slot = (blockIdx.x & 7) * (G >> 3) + (blockIdx.x >> 3);
  const int begin = split_begin(a.split, slot);
  const int end = split_begin(a.split, slot + 1);
  if (begin >= end) return;

  h8 wa[3][KR][OB];
  f4 bias4[OB];
  {
    const h8* wp = reinterpret_cast<const h8*>(a.w) + lane;
#pragma unroll
    for (int dy = 0; dy < 3; ++dy)
#pragma unroll
      for (int kc = 0; kc < KR; ++kc)
#pragma unroll
        for (int b = 0; b < OB; ++b) wa[dy][kc][b] = wp[((dy * KR + kc) * OB + b) * 64];
#pragma unroll
    for (int b = 0; b < OB; ++b)
      bias4[b] = *reinterpret_cast<const f4*>(a.bias + q * 4 * OB + 4 * b);
  }
  // The taps have landed before the first copy goes out: waits inside the loop
  // then count the loop's own memory instructions only.
  __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)

  const uint32_t rowb = (uint32_t)a.Wp * L::PXB;
  const uint32_t img = (uint32_t)a.Hp * rowb;
  const uint32_t lds0 = lds_byte_addr(rlds);
  // B read of tile t, product kc: byte rb[.] + 16 * PXB * t (+ 64 * kc unswizzled).
  int rb[SWZ ? KR : 1];
  if constexpr (SWZ) {
#pragma unroll
    for (int kc = 0; kc < KR; ++kc) rb[kc] = (j + kc) * L::PXB + ((q ^ (((j + kc) >> 1) & 2)) << 4);
  } else {
    rb[0] = j * L::PXB + 16 * q;
  }
  const uint32_t vmask = L::VO == 4 || q < L::VO ? ~0u : 0u;
  // Staging of this lane's channels [4 OB q, 4 OB q + 4 OB) of pixel j.
  const int mb = a.M * 2;
  const int sw = L::STG + j * mb + q * 8 * OB;

  int n = 0, sg = 0, y0 = 0;
  __amdgpu_buffer_rsrc_t rs;
  uint32_t doff[NI];  // copies' byte offsets from the start of a padded row
  for (int it = begin; it < end;) {
    {
      const uint32_t t = fdiv((uint32_t)it, a.fd_H);
      y0 = it - (int)(t * (uint32_t)a.H);
      const uint32_t nn = fdiv(t, a.fd_seg);
      sg = (int)(t - nn * (uint32_t)a.n_seg);
      n = (int)nn;
    }
    const int len = min(end - it, a.H - y0);
    const int x0 = sg * a.seg_w;
    const int valid = min(a.seg_w, a.W - x0);
    {
      const char* ib = reinterpret_cast<const char*>(a.in) + (int64_t)n * img;
      rs = __builtin_amdgcn_make_buffer_rsrc((void*)ib, (short)0, (int)img, 0x00020000);
    }
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int o = 1024 * i + 16 * lane;
      const int src = SWZ ? 1024 * i + (lane >> 2) * L::PXB + (((lane & 3) ^ ((lane >> 3) & 2)) << 4) : o;
      doff[i] = o < (valid + 2) * L::PXB ? (uint32_t)(x0 * L::PXB + src) : kOob;
    }
    // Input row r of the run (padded row y0 + r) into ring slot s.
    auto issue_row = [&](int r, int s) {
      const uint32_t ro = r <= len + 1 ? (uint32_t)(y0 + r) * rowb : kOob;  // uniform
#pragma unroll
      for (int i = 0; i < NI; ++i)
        dma16_buf(lds0 + (uint32_t)(s * L::SLOT + 1024 * i), rs, (doff[i] | ro) >= kOob ? kOob : doff[i] + ro);
    };
    // Output row k of the run as a buffer resource over the segment's pixels.
    auto out_row = [&](const uint16_t* base, int k) {
      const char* p = reinterpret_cast<const char*>(base) +
                      (((int64_t)n * a.Hp + y0 + k + 1) * a.Wp + x0 + 1) * mb;
      return __builtin_amdgcn_make_buffer_rsrc((void*)p, (short)0, k < len ? valid * mb : 0, 0x00020000);
    };
    auto issue_skips = [&](int k) {
#pragma unroll
      for (int e = 0; e < NSKIP; ++e) {
        const __amdgpu_buffer_rsrc_t rk = out_row(e == 0 ? a.skip0 : a.skip1, k);
#pragma unroll
        for (int i = 0; i < NS; ++i)
          dma16_buf(lds0 + (uint32_t)(L::STG + ((k & 1) * NSKIP + e) * L::SSLOT + 1024 * i), rk,
                    (uint32_t)(1024 * i + 16 * lane));
      }
    };

    if constexpr (NSKIP > 0) issue_skips(0);
#pragma unroll
    for (int r = 0; r < R - 1; ++r) issue_row(r, r);
    int s = 0;  // ring slot of input row k
#pragma unroll 1
    for (int k = 0; k < len; ++k) {
      // Input row k + 2 has landed (and with it rows k, k + 1).
      if (k >= LA)
        wait_vmcnt<(LA - 1) * (NI + NSK) + LA * NS>();
      else if (k == 0)
        wait_vmcnt<(LA - 1) * NI>();
      else
        wait_vmcnt<(LA - 1) * NI + NSK + NS>();
      static_assert(LA == 2, "the waits of rows 0 .. LA - 1");
      if constexpr (NSKIP > 0) issue_skips(k + 1);
      issue_row(k + R - 1, s == 0 ? R - 1 : s - 1);

      f4 acc[T][OB];
#pragma unroll
      for (int t = 0; t < T; ++t)
#pragma unroll
        for (int b = 0; b < OB; ++b) acc[t][b] = bias4[b];
      const char* row[3];
#pragma unroll
      for (int dy = 0; dy < 3; ++dy)
        row[dy] = rlds + (s + dy >= R ? s + dy - R : s + dy) * L::SLOT;
      rows_fold<L, OB>(wa, row, rb, vmask, acc);

      if constexpr (NSKIP > 0) wait_vmcnt<2 * NI + NS + NSK>();  // residual row k
      char* const st = rlds + sw + (NSKIP > 0 ? (k & 1) * NSKIP * L::SSLOT : 0);
      auto epilogue = [&](auto act_tag) {
        constexpr int ACT = decltype(act_tag)::value;
#pragma unroll
        for (int b = 0; b < OB; ++b)
          if (q * 4 * OB + 4 * b < a.M) {
#pragma unroll
            for (int t = 0; t < T; ++t) {
              char* p = st + t * 16 * mb + 8 * b;
              h4 r = strip_act4<ACT>(acc[t][b]);
#pragma unroll
              for (int e = 0; e < NSKIP; ++e) r += *reinterpret_cast<const h4*>(p + e * L::SSLOT);
              *reinterpret_cast<h4*>(p) = r;
            }
          }
      };
      if (a.act == kActRelu)
        epilogue(IntC<kActRelu>{});
      else if (a.act == kActSilu)
        epilogue(IntC<kActSilu>{});
      else
        epilogue(IntC<kActNone>{});
      const char* lin = rlds + L::STG + (NSKIP > 0 ? (k & 1) * NSKIP * L::SSLOT : 0) + 16 * lane;
      if (a.nt_out)
        rows_store<NS, kNonTemporal>(lin, out_row(a.out, k), lane);
      else
        rows_store<NS, 0>(lin, out_row(a.out, k), lane);
      s = s + 1 == R ? 0 : s + 1;
    }
    it += len;
  }
  wait_vmcnt<0>();  // no copy into LDS outlives the workgroup
}

// ---------------------------------------------------------------------------
// Head pair: 1 -> 32 head conv on the boundary input, then a 32 -> 32 conv
// ---------------------------------------------------------------------------
//
// conv3x3_rows whose ring rows are not copied from memory but computed: the head
// conv of one row (direct_conv_c1_mfma's product, channel order and epilogue,
// so the same bits as the two convs apart) goes straight into the ring, and its
// output tensor never exists. Step k computes head row k + 3 while it folds rows
// k .. k + 2; the input of the row after that is requested a step ahead. Head
// pixels outside the image are zero: the second conv's padding.
// No unit is the bound at 540x960 (matrix units 18% busy, LDS 20%, 1.6 TB/s
// written): the launch, and a wave's own chain a step (input, head product, LDS,
// nine folds, staging, stores) with two waves per SIMD over nine rows. Head and
// conv apart 11 + 17 us there, 21 here; the 32-channel model's frame 62.7 -> 54.7 us
// (with the tail still apart), at 2x1080x1920 390 -> 301.
struct HeadPairL : RowsL<32, 2, 0> {
  static constexpr int R = 4;
  static constexpr int STG = R * SLOT;
  static constexpr size_t lds_bytes() { return STG + SSLOT; }
};

// AUX: the output stores' cache policy (a branch between two kinds of stores
// would make the compiler's wait counts assume none).
template <int ACT1, int BIN, int AUX>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2)))
conv3x3_head_pair(HeadPairArgs a) {
  using L = HeadPairL;
  constexpr int T = L::T, KR = L::KR, NS = L::NS, R = L::R, OB = 2, NB = 2;
  constexpr int EB = BIN == 2 ? 4 : 2;  // bytes per input element
  extern __shared__ __attribute__((aligned(16))) char rlds[];
  const int lane = threadIdx.x;
  const int j = lane & 15;
  const int q = lane >> 4;

  const int G = gridDim.x;
  const int slot = (blockIdx.x & 7) * (G >> 3) + (blockIdx.x >> 3);
  const int begin = split_begin(a.r.split, slot);
  const int end = split_begin(a.r.split, slot + 1);
  if (begin >= end) return;

  h8 wa[3][KR][OB];
  f4 bias4[OB];
  h4 wh[NB];      // the head's taps, as in direct_conv_c1_mfma
  f4 hbias[NB];
  {
    const h8* wp = reinterpret_cast<const h8*>(a.r.w) + lane;
#pragma unroll
    for (int dy = 0; dy < 3; ++dy)
#pragma unroll
      for (int kc = 0; kc < KR; ++kc)
#pragma unroll
        for (int b = 0; b < OB; ++b) wa[dy][kc][b] = wp[((dy * KR + kc) * OB + b) * 64];
#pragma unroll
    for (int b = 0; b < OB; ++b) {
      bias4[b] = *reinterpret_cast<const f4*>(a.r.bias + q * 4 * OB + 4 * b);
      hbias[b] = *reinterpret_cast<const f4*>(a.bias1 + q * 4 * NB + 4 * b);
      const int ch = (j >> 2) * 4 * NB + 4 * b + (j & 3);  // A row j of block b
      const _Float16* tp = reinterpret_cast<const _Float16*>(a.w1) + ch * 10 + 3 * (q < 3 ? q : 0);
      wh[b] = q < 3 ? h4{tp[0], tp[1], tp[2], (_Float16)0.0f} : h4{0, 0, 0, 0};
    }
  }
  const int H = a.r.H, W = a.r.W;
  int rb[KR];
#pragma unroll
  for (int kc = 0; kc < KR; ++kc) rb[kc] = (j + kc) * L::PXB + ((q ^ (((j + kc) >> 1) & 2)) << 4);
  const int hw = j * L::PXB + ((q ^ ((j >> 1) & 2)) << 4);  // head pixel j, octet q
  constexpr int M = 32;
  const int sw = L::STG + j * M * 2 + q * 8 * OB;

  int n = 0, y0 = 0;
  const uint32_t img = (uint32_t)H * (uint32_t)W * EB;
  for (int it = begin; it < end;) {
    int sg;
    {
      const uint32_t t = fdiv((uint32_t)it, a.r.fd_H);
      y0 = it - (int)(t * (uint32_t)H);
      const uint32_t nn = fdiv(t, a.r.fd_seg);
      sg = (int)(t - nn * (uint32_t)a.r.n_seg);
      n = (int)nn;
    }
    const int len = min(end - it, H - y0);
    const int x0 = sg * a.r.seg_w;
    const int valid = min(a.r.seg_w, W - x0);
    const char* ib = reinterpret_cast<const char*>(a.r.in) + (int64_t)n * img;
    const __amdgpu_buffer_rsrc_t rs =
        __builtin_amdgcn_make_buffer_rsrc((void*)ib, (short)0, (int)img, 0x00020000);
    // Ring pixel p = 16 t + j is image column x0 - 1 + p; its taps the columns
    // x0 - 2 + p .. x0 + p, as byte offsets in a row (kOob outside the image).
    uint32_t coff[T][3];
    uint32_t cmask[T];
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const int x = x0 - 1 + 16 * t + j;
      cmask[t] = x >= 0 && x < W ? ~0u : 0u;
#pragma unroll
      for (int dx = 0; dx < 3; ++dx) {
        const int c = x - 1 + dx;
        coff[t][dx] = c >= 0 && c < W ? (uint32_t)c * EB : kOob;
      }
    }
    // Input of head row r of the run (image row y0 + r - 1): rows y0 + r - 2 + q.
    // Held as loaded, one value per register: head_row packs them behind an empty
    // asm statement, else the compiler packs them right after the request and so
    // waits there, a load's latency per step.
    uint32_t v[T][3];
    auto load_row = [&](int r, uint32_t (&v)[T][3]) {
      const int hr = y0 + r - 2 + q;
      const uint32_t ro = q < 3 && hr >= 0 && hr < H ? (uint32_t)hr * (uint32_t)W * EB : kOob;
#pragma unroll
      for (int t = 0; t < T; ++t)
#pragma unroll
        for (int dx = 0; dx < 3; ++dx) {
          const uint32_t o = (coff[t][dx] | ro) >= kOob ? kOob : coff[t][dx] + ro;
          if constexpr (BIN == 2)
            v[t][dx] = __builtin_amdgcn_raw_buffer_load_b32(rs, o, 0, 0);
          else
            v[t][dx] = __builtin_amdgcn_raw_buffer_load_b16(rs, o, 0, 0);
        }
    };
    auto head_row = [&](int r, int s, uint32_t (&v)[T][3]) {
      const int y = y0 + r - 1;
      const uint32_t rmask = y >= 0 && y < H ? ~0u : 0u;  // uniform
#pragma unroll
      for (int t = 0; t < T; ++t) {
        h4 bv = {0, 0, 0, 0};
#pragma unroll
        for (int dx = 0; dx < 3; ++dx) {
          uint32_t w = v[t][dx];
          asm volatile("" : "+v"(w));
          bv[dx] = BIN == 2 ? (_Float16)__builtin_bit_cast(float, w)
                            : __builtin_bit_cast(_Float16, (uint16_t)w);
        }
        const f4 z = {0, 0, 0, 0};
        const h4 zh = {0, 0, 0, 0};
        h4 o[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          const f4 d = __builtin_amdgcn_mfma_f32_16x16x16f16(wh[b], bv, z, 0, 0, 0) + hbias[b];
          o[b] = strip_act4<ACT1>(d) + zh;  // (+ 0 as fast4 adds absent residuals)
        }
        const u4 m = {rmask & cmask[t], rmask & cmask[t], rmask & cmask[t], rmask & cmask[t]};
        *reinterpret_cast<u4*>(rlds + s * L::SLOT + hw + 16 * L::PXB * t) =
            __builtin_bit_cast(u4, __builtin_shufflevector(o[0], o[1], 0, 1, 2, 3, 4, 5, 6, 7)) & m;
      }
    };
    {
      uint32_t p0[T][3], p1[T][3], p2[T][3];
      load_row(0, p0);
      load_row(1, p1);
      load_row(2, p2);
      load_row(3, v);
      head_row(0, 0, p0);
      head_row(1, 1, p1);
      head_row(2, 2, p2);
      // Dropped stores: the loop is entered with the memory instructions of its
      // back edge (a row's loads, then NS stores), so that its waits for the
      // loads leave the last step's stores in flight.
      rows_store<NS, AUX>(rlds + L::STG + 16 * lane,
                          __builtin_amdgcn_make_buffer_rsrc((void*)a.r.out, (short)0, 0, 0x00020000), lane);
    }
    int s = 0;  // ring slot of head row k
#pragma unroll 1
    for (int k = 0; k < len; ++k) {
      const char* row[3];
#pragma unroll
      for (int dy = 0; dy < 3; ++dy) row[dy] = rlds + ((s + dy) & (R - 1)) * L::SLOT;
      if (k + 1 < len) {  // uniform
        head_row(k + 3, (s + 3) & (R - 1), v);
        load_row(k + 4, v);
      }
      f4 acc[T][OB];
#pragma unroll
      for (int t = 0; t < T; ++t)
#pragma unroll
        for (int b = 0; b < OB; ++b) acc[t][b] = bias4[b];
      rows_fold<L, OB>(wa, row, rb, ~0u, acc);
      auto epilogue = [&](auto act_tag) {
        constexpr int ACT = decltype(act_tag)::value;
#pragma unroll
        for (int t = 0; t < T; ++t) {
          const h4 r0 = strip_act4<ACT>(acc[t][0]), r1 = strip_act4<ACT>(acc[t][1]);
          *reinterpret_cast<h8*>(rlds + sw + t * 16 * M * 2) =
              __builtin_shufflevector(r0, r1, 0, 1, 2, 3, 4, 5, 6, 7);
        }
      };
      if (a.r.act == kActRelu)
        epilogue(IntC<kActRelu>{});
      else if (a.r.act == kActSilu)
        epilogue(IntC<kActSilu>{});
      else
        epilogue(IntC<kActNone>{});
      const char* p = reinterpret_cast<const char*>(a.r.out) +
                      (((int64_t)n * a.r.Hp + y0 + k + 1) * a.r.Wp + x0 + 1) * (M * 2);
      rows_store<NS, AUX>(rlds + L::STG + 16 * lane,
                          __builtin_amdgcn_make_buffer_rsrc((void*)p, (short)0, valid * M * 2, 0x00020000), lane);
      s = (s + 1) & (R - 1);
    }
    it += len;
  }
}

// ---------------------------------------------------------------------------
// Tail pair: 32 -> 32 conv, then the 32 -> 4 tail conv with DepthToSpace(2)
// ---------------------------------------------------------------------------
//
// conv3x3_rows whose output rows t do not leave: they go into a second LDS ring
// (fp16, zero outside the image, which is the tail's padding), and the tail conv
// reads them from there. Each row is read from LDS once and multiplied by the
// taps of all three kernel rows, onto the sums of three output rows (conv3x3_rows
// reads it three times, which here bound the kernel by its LDS reads: the frame
// below took 48.1 and 128 us).
// Step i takes input row i, which completes t row i - 2, and t row i - 3, which
// completes output row i - 5. The tail's nine taps are K = 32 products like the
// conv's, of which only four rows of A hold a channel (0, 1 in rows 0, 1 and 2, 3
// in rows 4, 5, taken from the packed taps of conv3x3_tail), so lane (q, j),
// q < 2, ends with the two values of output row 2 y + q at pixel 2 x: one store
// per tile, bias, activation and Clip in fp32 before it.
// Every step issues NI copies (LA rows ahead) and NST stores.
// At 540x960 a run is 14 steps for nine rows, and no unit is the bound (25 us;
// matrix units 34% busy, LDS 12%, 2 TB/s): the launch and a wave's own chain a step,
// two waves per SIMD. The 32-channel model's frame with conv and tail apart and in
// one launch: 54.3 -> 47.2 us at 540x960, 155.7 -> 121 at 1080p, 300 -> 220 at
// 2x1080x1920.
struct TailPairL : RowsL<32, 2, 0> {
  static constexpr int OPX = IPX - 4;  // output pixels per segment, at most
  static constexpr int LA = 3;
  static constexpr int R = LA + 1;     // input ring slots
  static constexpr int TR = R * SLOT;  // two t slots
  static constexpr size_t lds_bytes() { return TR + 2 * SLOT + 256; }  // reads run 128 bytes past a slot
};

// PACK: the output is aligned for two-element stores.
template <int ACT1, bool F32, bool PACK>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2)))
conv3x3_tail_pair(TailPairArgs a) {
  using L = TailPairL;
  constexpr int T = L::T, KR = L::KR, NI = L::NI, LA = L::LA, R = L::R, OB = 2;
  constexpr int NST = PACK ? T : 2 * T;
  constexpr int EB = F32 ? 4 : 2;  // bytes per output element
  static_assert(LA == 3 && R == 4, "the waits of steps 0 .. LA - 1, slots by mask");
  extern __shared__ __attribute__((aligned(16))) char rlds[];
  const int lane = threadIdx.x;
  const int j = lane & 15;
  const int q = lane >> 4;

  const int G = gridDim.x;
  const int slot = (blockIdx.x & 7) * (G >> 3) + (blockIdx.x >> 3);
  const int begin = split_begin(a.r.split, slot);
  const int end = split_begin(a.r.split, slot + 1);
  if (begin >= end) return;

  h8 wa[3][KR][OB];
  h8 wt[3][KR][1];  // the tail's taps
  f4 bias4[OB];
  float tb[2];
  {
    const h8* wp = reinterpret_cast<const h8*>(a.r.w) + lane;
#pragma unroll
    for (int dy = 0; dy < 3; ++dy)
#pragma unroll
      for (int kc = 0; kc < KR; ++kc)
#pragma unroll
        for (int b = 0; b < OB; ++b) wa[dy][kc][b] = wp[((dy * KR + kc) * OB + b) * 64];
#pragma unroll
    for (int b = 0; b < OB; ++b) bias4[b] = *reinterpret_cast<const f4*>(a.r.bias + q * 4 * OB + 4 * b);
    // Packed as [dy][lane (q, dx * 4 + n)][8] (conv3x3_tail's B operand).
    const bool live = (j & 3) < 2 && j < 6;
    const int ch = 2 * (j >> 2) + (j & 1);
#pragma unroll
    for (int dy = 0; dy < 3; ++dy)
#pragma unroll
      for (int dx = 0; dx < 3; ++dx) {
        const h8 v = reinterpret_cast<const h8*>(a.w2)[dy * 64 + 16 * q + dx * 4 + (live ? ch : 0)];
        wt[dy][dx][0] = live ? v : h8{0, 0, 0, 0, 0, 0, 0, 0};
      }
    tb[0] = a.bias2[2 * (q & 1)];
    tb[1] = a.bias2[2 * (q & 1) + 1];
  }
  const int H = a.r.H, W = a.r.W;
  const uint32_t rowb = (uint32_t)a.r.Wp * L::PXB;
  const uint32_t img = (uint32_t)a.r.Hp * rowb;
  const uint32_t lds0 = lds_byte_addr(rlds);
  int rb[KR];
#pragma unroll
  for (int kc = 0; kc < KR; ++kc) rb[kc] = (j + kc) * L::PXB + ((q ^ (((j + kc) >> 1) & 2)) << 4);
  const int tw = j * L::PXB + ((q ^ ((j >> 1) & 2)) << 4);  // t pixel j, octet q

  for (int it = begin; it < end;) {
    const uint32_t tt = fdiv((uint32_t)it, a.r.fd_H);
    const int y0 = it - (int)(tt * (uint32_t)H);
    const uint32_t nn = fdiv(tt, a.r.fd_seg);
    const int sg = (int)(tt - nn * (uint32_t)a.r.n_seg);
    const int n = (int)nn;
    const int len = min(end - it, H - y0);
    const int x0 = sg * a.r.seg_w;
    const int valid = min(a.r.seg_w, W - x0);
    const char* ib = reinterpret_cast<const char*>(a.r.in) + (int64_t)n * img;
    const __amdgpu_buffer_rsrc_t rs =
        __builtin_amdgcn_make_buffer_rsrc((void*)ib, (short)0, (int)img, 0x00020000);
    char* const ob = reinterpret_cast<char*>(a.r.out) + (int64_t)n * 4 * H * W * EB;
    const __amdgpu_buffer_rsrc_t ro =
        __builtin_amdgcn_make_buffer_rsrc((void*)ob, (short)0, (int)((uint32_t)4 * H * W * EB), 0x00020000);
    // Ring pixel i is padded column x0 - 1 + i, t pixel p image column x0 - 1 + p.
    uint32_t doff[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int px = (1024 / L::PXB) * i + (lane >> 2);
      const int col = x0 - 1 + px;
      const uint32_t src = (uint32_t)(col * L::PXB + (((lane & 3) ^ ((lane >> 3) & 2)) << 4));
      doff[i] = col >= 0 && col < a.r.Wp && px < valid + 4 ? src : kOob;
    }
    uint32_t cmask[T], ooff[T];
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const int x = x0 - 1 + 16 * t + j;
      cmask[t] = x >= 0 && x < W ? ~0u : 0u;
      const int o = 16 * t + j;
      ooff[t] = q < 2 && o < valid ? (uint32_t)(q * 2 * W + 2 * (x0 + o)) * EB : kOob;
    }
    // Input row i of the run (padded row y0 - 1 + i) into ring slot s.
    auto issue_row = [&](int i, int s) {
      const int pr = y0 - 1 + i;
      const uint32_t rofs = pr >= 0 && pr < a.r.Hp && i <= len + 3 ? (uint32_t)pr * rowb : kOob;  // uniform
#pragma unroll
      for (int c = 0; c < NI; ++c)
        dma16_buf(lds0 + (uint32_t)(s * L::SLOT + 1024 * c), rs, (doff[c] | rofs) >= kOob ? kOob : doff[c] + rofs);
    };
#pragma unroll
    for (int i = 0; i < LA; ++i) issue_row(i, i);
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): the taps, see conv3x3_rows
    // Sums of three rows each: A[2] the oldest, completed by this step's row.
    const f4 z = {0, 0, 0, 0};
    f4 A[3][T][OB], O[3][T][1];
#pragma unroll
    for (int t = 0; t < T; ++t) {
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        A[d][t][0] = A[d][t][1] = z;
        O[d][t][0] = z;
      }
    }
#pragma unroll 1
    for (int i = 0; i < len + 5; ++i) {
      // Input row i has landed.
      if (i >= LA)
        wait_vmcnt<(LA - 1) * NI + LA * NST>();
      else if (i == 0)
        wait_vmcnt<(LA - 1) * NI>();
      else if (i == 1)
        wait_vmcnt<(LA - 1) * NI + NST>();
      else
        wait_vmcnt<(LA - 1) * NI + 2 * NST>();
      issue_row(i + LA, (i + LA) & (R - 1));
      // Output row i - 5 from t rows up to i - 3, in the slot of the step before.
#pragma unroll
      for (int t = 0; t < T; ++t) {
        O[2][t][0] = O[1][t][0];
        O[1][t][0] = O[0][t][0];
        O[0][t][0] = z;
      }
      rows_fold_once<L, 1>(wt, rlds + L::TR + ((i + 1) & 1) * L::SLOT, rb, O);
      if (i < len + 4) {  // uniform: t row i - 2
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
          for (int b = 0; b < OB; ++b) {
            A[2][t][b] = A[1][t][b];
            A[1][t][b] = A[0][t][b];
            A[0][t][b] = bias4[b];
          }
        rows_fold_once<L, OB>(wa, rlds + (i & (R - 1)) * L::SLOT, rb, A);
        const int y = y0 + i - 3;
        const uint32_t rmask = y >= 0 && y < H ? ~0u : 0u;  // uniform
#pragma unroll
        for (int t = 0; t < T; ++t) {
          const h4 r0 = strip_act4<ACT1>(A[2][t][0]), r1 = strip_act4<ACT1>(A[2][t][1]);
          const u4 m = {rmask & cmask[t], rmask & cmask[t], rmask & cmask[t], rmask & cmask[t]};
          *reinterpret_cast<u4*>(rlds + L::TR + (i & 1) * L::SLOT + tw + 16 * L::PXB * t) =
              __builtin_bit_cast(u4, __builtin_shufflevector(r0, r1, 0, 1, 2, 3, 4, 5, 6, 7)) & m;
        }
      }
      const uint32_t orow = i >= 5 ? (uint32_t)(y0 + i - 5) * (uint32_t)(4 * W) * EB : kOob;  // uniform
#pragma unroll
      for (int t = 0; t < T; ++t) {
        float v[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          v[e] = apply_act(O[2][t][0][e] + tb[e], a.act2);
          if (a.do_clip) v[e] = apply_clip(v[e], a.clip_lo, a.clip_hi);
        }
        const uint32_t off = (ooff[t] | orow) >= kOob ? kOob : ooff[t] + orow;
        if constexpr (F32) {
          const u2 b = {__builtin_bit_cast(uint32_t, v[0]), __builtin_bit_cast(uint32_t, v[1])};
          if constexpr (PACK) {
            __builtin_amdgcn_raw_buffer_store_b64(b, ro, off, 0, 0);
          } else {
            __builtin_amdgcn_raw_buffer_store_b32(b[0], ro, off, 0, 0);
            __builtin_amdgcn_raw_buffer_store_b32(b[1], ro, off + 4, 0, 0);
          }
        } else {
          const _Float16 b0 = (_Float16)v[0], b1 = (_Float16)v[1];
          if constexpr (PACK) {
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, h2{b0, b1}), ro, off, 0, 0);
          } else {
            __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(uint16_t, b0), ro, off, 0, 0);
            __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(uint16_t, b1), ro, off + 2, 0, 0);
          }
        }
      }
    }
    it += len;
  }
  wait_vmcnt<0>();  // no copy into LDS outlives the workgroup
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

// Two tiles a step at C = 24 and 40, for more than 32 outputs: without a residual
// input at C = 40, where the taps and sums of four spill (40 -> 40 at 361x481 16.9
// against 11.6 us, 1080p 115 and 73; winograd_conv 24 and 259), and on up to 2^15
// pixels, where a launch is one short run a wave and four tiles make it longer
// (24 -> 40 + two residuals at 16x16 4.6 and 3.6 us, 100x160 5.0 and 4.2, 300x64 5.4
// and 4.5; winograd_conv 4.0, 4.3, 4.9). Above, four are up to 17% faster on runs of
// one row (200x300: 6.3 and 7.4).
constexpr bool rows_two_tiles(int C, int M, int nskip, int64_t pixels) {
  return C % 16 != 0 && M > 32 && (pixels <= 1 << 15 || (C == 40 && nskip == 0));
}

struct RowsPick {
  RowKernel fn = nullptr;
  size_t lds = 0;
  int seg = 0;  // output pixels per segment, at most
};

template <int C, int OB, int NSKIP>
RowsPick rows_pick(bool two) {
  auto of = [](auto tiles) {
    using L = RowsL<C, OB, NSKIP, decltype(tiles)::value>;
    return RowsPick{conv3x3_rows<C, OB, NSKIP, decltype(tiles)::value>, L::lds_bytes(), L::OPX};
  };
  if constexpr (C % 16 == 0 || rows_two_tiles(C, 16 * OB, NSKIP, (int64_t)1 << 40))
    return of(IntC<2>{});
  else if constexpr (!rows_two_tiles(C, 16 * OB, NSKIP, 1))
    return of(IntC<4>{});
  else
    return two ? of(IntC<2>{}) : of(IntC<4>{});
}

template <int C, int OB>
RowsPick rows_pick(int nskip, bool two) {
  return nskip == 0 ? rows_pick<C, OB, 0>(two) : nskip == 1 ? rows_pick<C, OB, 1>(two) : rows_pick<C, OB, 2>(two);
}

template <int C>
RowsPick rows_pick(int M, int nskip, int64_t pixels) {
  const bool two = rows_two_tiles(C, M, nskip, pixels);
  return M <= 16   ? rows_pick<C, 1>(nskip, two)
         : M <= 32 ? rows_pick<C, 2>(nskip, two)
                   : rows_pick<C, 3>(nskip, two);
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
  a.seg_w = (w.W + a.n_seg - 1) / a.n_seg;
  a.n_items = (int32_t)((int64_t)w.N * a.n_seg * w.H);
  a.fd_H = make_fastdiv((uint32_t)w.H);
  a.fd_seg = make_fastdiv((uint32_t)a.n_seg);
  return a;
}

// Grid of a launch (at most `cap` workgroups per CU) and its ranges in a.split.
template <class Args>
hipError_t rows_grid(void (*fn)(Args), DirectRowArgs& a, int threads, size_t lds, int cap, int fill, unsigned* blocks) {
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
  int64_t grid = (int64_t)cu_count() * (occ < cap ? occ : cap);
  if (grid > a.n_items) grid = a.n_items;
  grid = (grid + 7) / 8 * 8;
  a.split = make_split(a.n_items, (int)grid, a.H, fill);
  *blocks = (unsigned)grid;
  return hipSuccess;
}

// Outputs of up to 96 MiB are stored plainly: the next layer finds them in the
// last-level cache (32-channel model: 61 us at 540x960, 65 with non-temporal
// stores; 91 and 98 at 720p). Larger ones carry the hint (183 against 185 us at
// 1080p, 326 against 354 at 1440x2560, a lone 32 -> 32 conv with a residual at
// 1080p 65 against 86).
bool nt_stores(const DirectRowArgs& a) {
  return (int64_t)a.N * a.Hp * a.Wp * a.M * 2 > ((int64_t)96 << 20);
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
  DirectRowArgs a = row_args(w, 64);
  const RowKernel fn = w.C == 2   ? head_kernel<2>(w.M, a.act)
                       : w.C == 3 ? head_kernel<3>(w.M, a.act)
                                  : head_kernel<4>(w.M, a.act);
  const size_t lds = (size_t)4 * 16 * w.M * 2;
  unsigned blocks = 0;
  const hipError_t e = rows_grid(fn, a, 256, lds, 8, 0, &blocks);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(fn, dim3(blocks), dim3(256), lds, s, a);
  return hipGetLastError();
}

bool conv_rows_eligible(const WinoArgs& w) {
  const int64_t cm = w.C > w.M ? w.C : w.M;
  return inner_epilogue(w) && direct_rows_shape(w.C, w.M) && aligned16(w.in) &&
         aligned16(w.epi.out) && aligned16(w.epi.skip0) && aligned16(w.epi.skip1) &&
         fits32(w.N, w.H, w.W, cm, RowsL<16, 1, 0>::OPX);  // (the shorter segment)
}

hipError_t launch_conv_rows(const WinoArgs& w, hipStream_t s) {
  if (!conv_rows_eligible(w)) return hipErrorInvalidValue;
  const int nskip = (w.epi.skip0 != nullptr) + (w.epi.skip1 != nullptr);
  const int64_t pixels = (int64_t)w.N * w.H * w.W;
  RowsPick k;
  switch (w.C) {
    case 16: k = rows_pick<16>(w.M, nskip, pixels); break;
    case 24: k = rows_pick<24>(w.M, nskip, pixels); break;
    case 32: k = rows_pick<32>(w.M, nskip, pixels); break;
    case 40: k = rows_pick<40>(w.M, nskip, pixels); break;
    case 48: k = rows_pick<48>(w.M, nskip, pixels); break;
    default: return hipErrorInvalidValue;
  }
  DirectRowArgs a = row_args(w, k.seg);
  a.nt_out = nt_stores(a);
  // Eight waves per CU at most: more make the runs shorter (two rows of halo
  // each) without streaming faster (32 -> 32 + residual at 1080p: 94 us with
  // twelve, 86 with eight, 84 with five; 16 -> 16 at 1080p: 24, 26, 36).
  unsigned blocks = 0;
  const hipError_t e = rows_grid(k.fn, a, 64, k.lds, 8, 1, &blocks);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k.fn, dim3(blocks), dim3(64), k.lds, s, a);
  return hipGetLastError();
}

// The conv alone would run conv3x3_rows, and the head direct_conv_c1_mfma on the
// boundary input: the pair gives the same bits as the two.
bool head_pair_eligible(int64_t N, int64_t H, int64_t W, bool fp32) {
  return fits32(N, H, W, 32, HeadPairL::OPX) && head_reads_boundary_input(N, H, W, 32, fp32);
}

hipError_t launch_head_pair(const DirectArgs& head, const WinoArgs& conv, hipStream_t s) {
  if (!head_pair_eligible(head.N, head.H, head.W, head.in_kind == 2) || head.in_kind == 0 || head.M != 32 ||
      conv.C != 32 || conv.M != 32 || !inner_epilogue(conv) || conv.epi.skip0 != nullptr ||
      conv.epi.skip1 != nullptr || !aligned16(conv.epi.out))
    return hipErrorInvalidValue;
  HeadPairArgs a{};
  a.r = row_args(conv, HeadPairL::OPX);
  a.r.in = static_cast<const uint16_t*>(head.in);
  a.r.nt_out = nt_stores(a.r);
  a.w1 = head.w;
  a.bias1 = head.epi.bias;
  using Fn = void (*)(HeadPairArgs);
  auto pick = [&](auto bin_tag, auto aux_tag) -> Fn {
    constexpr int BIN = decltype(bin_tag)::value, AUX = decltype(aux_tag)::value;
    return head.epi.act == kActRelu   ? conv3x3_head_pair<kActRelu, BIN, AUX>
           : head.epi.act == kActSilu ? conv3x3_head_pair<kActSilu, BIN, AUX>
                                      : conv3x3_head_pair<kActNone, BIN, AUX>;
  };
  const bool f32 = head.in_kind == 2;
  const Fn fn = a.r.nt_out ? (f32 ? pick(IntC<2>{}, IntC<kNonTemporal>{}) : pick(IntC<1>{}, IntC<kNonTemporal>{}))
                           : (f32 ? pick(IntC<2>{}, IntC<0>{}) : pick(IntC<1>{}, IntC<0>{}));
  unsigned blocks = 0;
  const hipError_t e = rows_grid(fn, a.r, 64, HeadPairL::lds_bytes(), 8, 2, &blocks);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(fn, dim3(blocks), dim3(64), HeadPairL::lds_bytes(), s, a);
  return hipGetLastError();
}

// The conv alone would run conv3x3_rows and the tail conv3x3_tail.
bool tail_pair_eligible(int64_t N, int64_t H, int64_t W, bool fp32) {
  const int64_t out = 4 * H * W * (fp32 ? 4 : 2);
  return fits32(N, H, W, 32, TailPairL::OPX) && out < (int64_t)1 << 31;
}

hipError_t launch_tail_pair(const WinoArgs& conv, const WinoArgs& tail, hipStream_t s) {
  const bool f32 = tail.epi.out_kind == kOutNchwF32;
  if (!tail_pair_eligible(conv.N, conv.H, conv.W, f32) || conv.C != 32 || conv.M != 32 || tail.C != 32 ||
      tail.M != 4 || tail.epi.dts_b != 2 || (!f32 && tail.epi.out_kind != kOutNchwF16) ||
      conv.epi.skip0 != nullptr || conv.epi.skip1 != nullptr || tail.epi.skip0 != nullptr ||
      tail.epi.skip1 != nullptr || conv.epi.do_clip || !aligned16(conv.in))
    return hipErrorInvalidValue;
  TailPairArgs a{};
  a.r = row_args(conv, TailPairL::OPX);
  a.r.out = static_cast<uint16_t*>(tail.epi.out);
  a.w2 = tail.u + winograd_u_halfs(32, 4);
  a.bias2 = tail.epi.bias;
  a.act2 = tail.epi.act;
  a.do_clip = tail.epi.do_clip;
  a.clip_lo = tail.epi.clip_lo;
  a.clip_hi = tail.epi.clip_hi;
  using Fn = void (*)(TailPairArgs);
  auto pick = [&](auto f32_tag, auto pack_tag) -> Fn {
    constexpr bool F = decltype(f32_tag)::value != 0, P = decltype(pack_tag)::value != 0;
    return conv.epi.act == kActRelu   ? conv3x3_tail_pair<kActRelu, F, P>
           : conv.epi.act == kActSilu ? conv3x3_tail_pair<kActSilu, F, P>
                                      : conv3x3_tail_pair<kActNone, F, P>;
  };
  const bool pack = reinterpret_cast<uintptr_t>(tail.epi.out) % (f32 ? 8 : 4) == 0;
  const Fn fn = f32 ? (pack ? pick(IntC<1>{}, IntC<1>{}) : pick(IntC<1>{}, IntC<0>{}))
                    : (pack ? pick(IntC<0>{}, IntC<1>{}) : pick(IntC<0>{}, IntC<0>{}));
  unsigned blocks = 0;
  const hipError_t e = rows_grid(fn, a.r, 64, TailPairL::lds_bytes(), 8, 4, &blocks);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(fn, dim3(blocks), dim3(64), TailPairL::lds_bytes(), s, a);
  return hipGetLastError();
}

}  // namespace arthip
