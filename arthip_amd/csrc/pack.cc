#include "pack.h"

#include <cstring>

#include "half.h"

namespace arthip {

bool narrow_eligible(int C, int M) { return C % 32 == 0 && C <= 96 && M >= 1 && M <= 16; }

bool narrow_row_packed(int M) { return M >= 1 && 3 * M <= 16; }

size_t narrow_packed_halfs(int C, int M) {
  if (!narrow_eligible(C, M)) return 0;
  return static_cast<size_t>(narrow_row_packed(M) ? 3 : 9) * (C / 32) * 64 * 8;
}

size_t winograd_u_halfs(int C, int M) {
  const WinoGeom g = winograd_geom(C, M);
  return static_cast<size_t>(g.n_ob) * 16 * g.kc * 64 * 8;
}

size_t block_u_halfs(int C, int M) {
  const bool rows = C == M && (C == 64 || C == 96);
  return rows ? static_cast<size_t>(M / 16) * 12 * (C / 32) * 64 * 8 : 0;
}

size_t block_u_offset(int C, int M) { return winograd_u_halfs(C, M) + narrow_packed_halfs(C, M); }

bool direct_head_shape(int C, int M) {
  return C >= 2 && C <= 4 && (M == 32 || M == 64 || M == 96);
}

bool direct_rows_shape(int C, int M) {
  return C % 8 == 0 && C >= 16 && C <= 48 && M % 8 == 0 && M >= 8 && M <= 48;
}

size_t direct_rows_halfs(int C, int M) {
  if (direct_head_shape(C, M)) return static_cast<size_t>(M / 16) * 64 * 16;
  if (direct_rows_shape(C, M)) return static_cast<size_t>(3 * ((3 * C + 31) / 32)) * ((M + 15) / 16) * 64 * 8;
  return 0;
}

size_t direct_rows_offset(int C, int M) { return block_u_offset(C, M) + block_u_halfs(C, M); }

size_t winograd_packed_halfs(int C, int M) {
  return direct_rows_offset(C, M) + direct_rows_halfs(C, M);
}

// Direct taps of a narrow layer (layout in pack.h); `out` is zero-filled.
static void direct_rows_pack(const float* w, int M, int C, uint16_t* out) {
  const int n_ob = (M + 15) / 16;
  const int kr = (3 * C + 31) / 32;
  const bool head = direct_head_shape(C, M);
  for (int m = 0; m < M; ++m) {
    const int b = m % (4 * n_ob) / 4, i = m / (4 * n_ob) * 4 + m % 4;  // A row i of block b
    const float* wm = w + static_cast<size_t>(m) * C * 9;
    for (int dy = 0; dy < 3; ++dy) {
      // Value k = dx * C + c of the row at slot q = k / 8 (of four per product), k % 8.
      uint16_t* const row = head ? out + (static_cast<size_t>(b) * 64 + dy * 16 + i) * 16
                                 : out + ((static_cast<size_t>(dy) * kr * n_ob + b) * 64 + i) * 8;
      int k = 0;
      for (int dx = 0; dx < 3; ++dx)
        for (int c = 0; c < C; ++c, ++k) {
          const size_t at = head ? static_cast<size_t>(k)
                                 : static_cast<size_t>(k >> 5) * n_ob * 512 + ((k >> 3) & 3) * 128 + (k & 7);
          row[at] = f32_to_f16(wm[c * 9 + dy * 3 + dx]);
        }
    }
  }
}

void winograd_pack(const float* w, int M, int C, uint16_t* out) {
  const WinoGeom g = winograd_geom(C, M);
  const size_t total = winograd_packed_halfs(C, M);
  std::memset(out, 0, total * sizeof(uint16_t));
  if (narrow_eligible(C, M)) {
    uint16_t* nb = out + winograd_u_halfs(C, M);
    const int kcn = C / 32;
    const bool rows = narrow_row_packed(M);
    for (int n = 0; n < M; ++n)
      for (int c = 0; c < C; ++c)
        for (int t = 0; t < 9; ++t) {
          const int kc = c / 32, q = (c % 32) / 8, e = c % 8;
          const int slot = rows ? t / 3 : t;             // B operand index
          const int col = rows ? (t % 3) * M + n : n;    // B column
          const size_t idx = ((static_cast<size_t>(slot) * kcn + kc) * 64 + col + 16 * q) * 8 + e;
          nb[idx] = f32_to_f16(w[(static_cast<size_t>(n) * C + c) * 9 + t]);
        }
  }
  // G = [[1,0,0],[1/2,1/2,1/2],[1/2,-1/2,1/2],[0,0,1]]; U = G g G^T in double,
  // scaled by 4 (exact), rounded once to fp16.
  static const double G[4][3] = {{1, 0, 0}, {0.5, 0.5, 0.5}, {0.5, -0.5, 0.5}, {0, 0, 1}};
  if (block_u_halfs(C, M) != 0) {
    // Row filters of the fused block: U_dy[p] = G[p] . w[dy][0..2], rounded once.
    uint16_t* bu = out + block_u_offset(C, M);
    const int kcn = C / 32;
    for (int m = 0; m < M; ++m) {
      const int ob = m / 16, row = m % 16;
      for (int c = 0; c < C; ++c) {
        const float* k = w + (static_cast<size_t>(m) * C + c) * 9;
        const int kc = c / 32, kk = c % 32;
        const int lane = row + 16 * (kk / 8), e = kk % 8;
        for (int dy = 0; dy < 3; ++dy)
          for (int p = 0; p < 4; ++p) {
            const double u = G[p][0] * k[dy * 3] + G[p][1] * k[dy * 3 + 1] + G[p][2] * k[dy * 3 + 2];
            const size_t idx =
                ((((static_cast<size_t>(ob) * 3 + dy) * 4 + p) * kcn + kc) * 64 + lane) * 8 + e;
            bu[idx] = f32_to_f16(static_cast<float>(u));
          }
      }
    }
  }
  if (direct_rows_halfs(C, M) != 0) direct_rows_pack(w, M, C, out + direct_rows_offset(C, M));
  for (int m = 0; m < M; ++m) {
    const int ob = m / 16, row = m % 16;
    for (int c = 0; c < C; ++c) {
      const float* k = w + (static_cast<size_t>(m) * C + c) * 9;
      double Gg[4][3];
      for (int i = 0; i < 4; ++i)
        for (int j = 0; j < 3; ++j)
          Gg[i][j] = G[i][0] * k[0 * 3 + j] + G[i][1] * k[1 * 3 + j] + G[i][2] * k[2 * 3 + j];
      const int kc = c / 32, kk = c % 32;
      const int lane = row + 16 * (kk / 8), e = kk % 8;
      for (int i = 0; i < 4; ++i)
        for (int j = 0; j < 4; ++j) {
          const double u = Gg[i][0] * G[j][0] + Gg[i][1] * G[j][1] + Gg[i][2] * G[j][2];
          const int p = i * 4 + j;
          const size_t idx = ((((static_cast<size_t>(ob) * 16 + p) * g.kc + kc) * 64) + lane) * 8 + e;
          out[idx] = f32_to_f16(static_cast<float>(4.0 * u));
        }
    }
  }
}

size_t direct_packed_halfs(int M) { return static_cast<size_t>(direct_g8(M)) * 8 * 5 * 2; }

void direct_pack(const float* w, int M, uint16_t* out) {
  const size_t total = direct_packed_halfs(M);
  std::memset(out, 0, total * sizeof(uint16_t));
  for (int m = 0; m < M; ++m) {
    const int g = m / 8, c = m % 8;
    for (int t = 0; t < 9; ++t) {
      const size_t idx = ((static_cast<size_t>(g) * 8 + c) * 5 + t / 2) * 2 + (t % 2);
      out[idx] = f32_to_f16(w[static_cast<size_t>(m) * 9 + t]);
    }
  }
}

size_t bias_padded_len(int M) {
  size_t n = (static_cast<size_t>(M) + 15) / 16 * 16;
  const size_t d = static_cast<size_t>(direct_g8(M)) * 8;
  return n > d ? n : d;
}

void bias_pad(const float* bias, int M, float* out) {
  const size_t n = bias_padded_len(M);
  for (size_t i = 0; i < n; ++i) out[i] = (bias != nullptr && i < static_cast<size_t>(M)) ? bias[i] : 0.0f;
}

}  // namespace arthip
