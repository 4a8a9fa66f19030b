// The bandwidth yardstick of profiles/gla_chunk_config4_prompts.md: the loads and stores of gla_chunk_kernel without its arithmetic.
// One workgroup of four wavefronts per (prompt, head) walks its tokens in blocks of 32, loads of block n + 1 in front of the stores of
// block n, the wavefronts in step; heads of a token lie side by side, as in the layer. A block's 32 rows of q, k, v (256 bytes) and gate
// (512) are dealt to the wavefronts so that one load instruction finds LP 16-byte pieces of a row together, and a wavefront's 64 bytes
// of an output row are stored 4 SB bytes per instruction and row.
//   hipcc --offload-arch=gfx950 -O3 -std=c++17 -Xclang -target-feature -Xclang -packed-fp32-ops profiles/gla_prompt_copy.hip -o gla_prompt_copy
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <vector>

#define CHECK(x)                                                                     \
  do {                                                                               \
    const hipError_t e = (x);                                                        \
    if (e != hipSuccess) { printf("%s: %s\n", #x, hipGetErrorString(e)); exit(1); }  \
  } while (0)

constexpr int kPrompts = 16, kTokens = 8192, kHeads = 28, kBlock = 32;
static_assert(kTokens % kBlock == 0, "whole blocks");
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

struct Rows {
  u32x4 q[2], k[2], v[2], g[2][2];
};

// LP: 16-byte pieces of a row per load instruction (4, 8 or 16); SB: bytes a lane stores at a time (8 or 16)
template <int LP, int SB>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void copy_kernel(const char *q, const char *k, const char *v, const char *g, char *out) {
  const int b = blockIdx.x / kHeads, h = blockIdx.x % kHeads;
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  // this thread's two rows of a block and its piece of them: the wavefront has LP of a row's 16 pieces and 128 / LP of the 32 rows
  constexpr int kAcross = 16 / LP, kRowsOfWave = 128 / LP;
  const int piece = LP * (w % kAcross) + lane % LP, row = kRowsOfWave * (w / kAcross) + lane / LP * 2;
  const int64_t stride = kHeads * 256;   // of a token's 16-bit rows; its gates: twice that
  const int64_t first = (int64_t)b * kTokens * stride + h * 256;
  q += first + row * stride + piece * 16;
  k += first + row * stride + piece * 16;
  v += first + row * stride + piece * 16;
  g += 2 * (first + row * stride + piece * 16);
  out += first + w * 64 + (int64_t)(lane & 15) * stride + (lane >> 4) * SB;
  auto fetch = [&](Rows &x, int n) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int64_t at = (int64_t)(n * kBlock + u) * stride;
      x.q[u] = *reinterpret_cast<const u32x4 *>(q + at);
      x.k[u] = *reinterpret_cast<const u32x4 *>(k + at);
      x.v[u] = *reinterpret_cast<const u32x4 *>(v + at);
#pragma unroll
      for (int j = 0; j < 2; ++j) x.g[u][j] = *reinterpret_cast<const u32x4 *>(g + 2 * at + 16 * j);
    }
  };
  auto store = [&](const Rows &x, int n) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const u32x4 y = x.q[u] ^ x.k[u] ^ x.v[u] ^ x.g[u][0] ^ x.g[u][1];   // (16 bytes of each of two rows: all of a wavefront's output)
      char *at = out + (int64_t)(n * kBlock + 16 * u) * stride;
      if constexpr (SB == 16) {
        *reinterpret_cast<u32x4 *>(at) = y;
      } else {
        *reinterpret_cast<u32x2 *>(at) = y.xy;
        *reinterpret_cast<u32x2 *>(at + 32) = y.zw;
      }
    }
  };
  constexpr int kLast = kTokens / kBlock - 1;
  Rows x0, x1;
  fetch(x0, 0);
  for (int n = 0; n <= kLast; n += 2) {
    fetch(x1, min(n + 1, kLast));
    __syncthreads();
    store(x0, n);
    fetch(x0, min(n + 2, kLast));
    __syncthreads();
    store(x1, min(n + 1, kLast));
  }
}

int main() {
  const size_t row16 = (size_t)kPrompts * kTokens * kHeads * 256;
  char *q, *k, *v, *g, *out;
  CHECK(hipMalloc(&q, row16)); CHECK(hipMalloc(&k, row16)); CHECK(hipMalloc(&v, row16)); CHECK(hipMalloc(&g, 2 * row16)); CHECK(hipMalloc(&out, row16));
  for (char *x : {q, k, v, g}) CHECK(hipMemset(x, 17, x == g ? 2 * row16 : row16));
  hipEvent_t a, z;
  CHECK(hipEventCreate(&a)); CHECK(hipEventCreate(&z));
  auto time = [&](const char *what, auto kernel) {
    std::vector<float> ms;
    for (int i = 0; i < 12; ++i) {
      CHECK(hipEventRecord(a));
      hipLaunchKernelGGL(kernel, dim3(kPrompts * kHeads), dim3(256), 0, 0, q, k, v, g, out);
      CHECK(hipGetLastError());
      CHECK(hipEventRecord(z));
      CHECK(hipEventSynchronize(z));
      float t;
      CHECK(hipEventElapsedTime(&t, a, z));
      if (i >= 2) ms.push_back(t);
    }
    std::sort(ms.begin(), ms.end());
    printf("%-60s %8.1f us  %5.2f TB/s\n", what, 1e3 * ms[ms.size() / 2], 6.0 * row16 / ms[ms.size() / 2] * 1e-9);
    fflush(stdout);
  };
  time("loads of 64 bytes of 16 rows, stores of 32 bytes", copy_kernel<4, 8>);
  time("loads of 64 bytes of 16 rows, stores of 64 bytes", copy_kernel<4, 16>);
  time("loads of 128 bytes of 8 rows, stores of 64 bytes", copy_kernel<8, 16>);
  time("loads of whole rows (256 bytes) of 4, stores of 64 bytes", copy_kernel<16, 16>);
  return 0;
}
