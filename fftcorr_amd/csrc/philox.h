// Random catalogues come from a counter-based generator, Philox4x32-10 (Salmon,
// Moraes, Dror and Shaw, "Parallel random numbers: as easy as 1, 2, 3",
// SC 2011): 10 rounds of two 32x32->64-bit multiplies with the key bumped by
// the Weyl constants between rounds.  Particle i of stream `seed` uses the
// counters (i, 0, 0) and (i, 1, 0) -- two 4-word draws, six words -> three
// 53-bit uniforms -- so any range of particles can be generated
// independently and the catalogue is the same however it is batched.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace fc {

struct Philox {
  uint32_t c[4];
};

__host__ __device__ inline void mulhilo(uint32_t a, uint32_t b, uint32_t* hi, uint32_t* lo) {
  const uint64_t p = (uint64_t)a * b;
  *hi = (uint32_t)(p >> 32);
  *lo = (uint32_t)p;
}

__host__ __device__ inline Philox philox4x32_10(Philox x, uint32_t k0, uint32_t k1) {
  const uint32_t M0 = 0xD2511F53u, M1 = 0xCD9E8D57u;
  const uint32_t W0 = 0x9E3779B9u, W1 = 0xBB67AE85u;
  for (int r = 0; r < 10; ++r) {
    if (r > 0) {
      k0 += W0;
      k1 += W1;
    }
    uint32_t hi0, lo0, hi1, lo1;
    mulhilo(M0, x.c[0], &hi0, &lo0);
    mulhilo(M1, x.c[2], &hi1, &lo1);
    x = Philox{{hi1 ^ x.c[1] ^ k0, lo1, hi0 ^ x.c[3] ^ k1, lo0}};
  }
  return x;
}

// Uniform in [0, 1) from two words: 27 + 26 bits (53 in all).
__device__ __forceinline__ double u53(uint32_t a, uint32_t b) {
  return ((double)(a >> 5) * 67108864.0 + (double)(b >> 6)) * (1.0 / 9007199254740992.0);
}

// Particle `ctr` of stream `seed`: lo + u * span per axis.
__device__ __forceinline__ double3 random_uniform(const double3& lo, const double3& span,
                                                  uint64_t seed, uint64_t ctr) {
#pragma clang fp contract(off)
  const uint32_t c0 = (uint32_t)ctr, c1 = (uint32_t)(ctr >> 32);
  const uint32_t k0 = (uint32_t)seed, k1 = (uint32_t)(seed >> 32);
  const Philox a = philox4x32_10(Philox{{c0, c1, 0u, 0u}}, k0, k1);
  const Philox b = philox4x32_10(Philox{{c0, c1, 1u, 0u}}, k0, k1);
  return make_double3(lo.x + u53(a.c[0], a.c[1]) * span.x, lo.y + u53(a.c[2], a.c[3]) * span.y,
                      lo.z + u53(b.c[0], b.c[1]) * span.z);
}

}  // namespace fc
