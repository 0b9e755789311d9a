// Walks the addresses of the ring GEMM's A loads and of the one-block-ahead attention kernel's K and V^T
// loads (laya-cuda_amd/csrc/ranges.hpp) for operands of many sizes: scalar offsets stay inside the resource,
// rows and keys that exist are read from their own place, and V^T chunks never leave their head dim's row.
#include <cstdio>
#include <cstdlib>
#include <initializer_list>

#include "ranges.hpp"

static void require(bool ok, const char* what, int a, int b, int c) {
  if (ok) return;
  std::fprintf(stderr, "%s: %d %d %d\n", what, a, b, c);
  std::exit(1);
}

int main() {
  long long checked = 0;
  for (int k : {192, 768, 4096})
    for (int left = 1; left <= 300; ++left) {
      const unsigned row_bytes = 2u * k;
      const unsigned long long bytes = static_cast<unsigned long long>(left) * row_bytes;
      for (int slab = 0; slab < k / 64; ++slab)
        for (int q = 0; q < 4; ++q) {
          const unsigned long long soffset = slab * 128ull + laya::ring_row_offset(q, row_bytes, laya::ring_row_limit(left, row_bytes));
          require(soffset < bytes, "scalar offset past the A operand", k, left, q);
          for (int r = 0; r < 64; ++r) {
            if (64 * q + r >= left) continue;
            const unsigned long long at = static_cast<unsigned long long>(r) * row_bytes + soffset;
            require(at == static_cast<unsigned long long>(64 * q + r) * row_bytes + slab * 128ull && at + 128 <= bytes,
                    "an A row is read elsewhere", left, q, r);
            ++checked;
          }
        }
    }
  for (int m = 16; m <= 400; m += 16)
    for (int kb = 0; kb < m; kb += 16)
      for (int half = 0; half < 2; ++half) {
        const unsigned soffset = laya::key_half_offset(kb, half, m);
        require(soffset < static_cast<unsigned>(m) * 128u, "scalar offset past the K plane", m, kb, half);
        for (int c = 0; c < 8; ++c) {
          const int key = laya::value_chunk_key(kb, c, m);
          require(key >= 0 && key + 8 <= m, "a V^T chunk leaves its row", m, kb, c);
          if (kb + 8 * c + 8 <= m) require(key == kb + 8 * c, "a V^T chunk is read elsewhere", m, kb, c);
        }
        if (kb + 32 * half < m) require(soffset == (kb + 32u * static_cast<unsigned>(half)) * 128u, "a K half is read elsewhere", m, kb, half);
        ++checked;
      }
  std::printf("checked %lld\n", checked);
  return 0;
}
