// log1p in FP64 for non-negative arguments, with a table, for the statistics' inner loop.
//
// Tang's method (ACM TOMS 16(4), 1990): u = 1 + y = 2^k m with 1 <= m < 2, and with an 11-bit
// reciprocal 1/c of the middle of m's interval of 1/128, log u = k ln 2 + log c + log(1 + r),
// r = m / c - 1, |r| <= 1/128, log(1 + r) as its series to r^8 (the next term is below 2^-59
// of the sum).  c = 1 for the first interval, so a small y comes out as y - y^2/2 + ... with
// nothing cancelled, and no term is negative before it.  What 1 + y rounds away goes into r;
// ln 2 and log c have a high part on a grid of 2^-42, so that k ln2 + log c is exact.
// The head of r is kept apart from that rest, which would otherwise round it.
// Against 80-bit arithmetic, 4 million arguments a range: at most 0.75 units in the last place
// from 1e-300 to 1e300, rms 0.289 (a host's log1p: 0.83, 0.306).  About 40 instructions.
#pragma once
#include <cstdint>

#if defined(__HIPCC__)
#define SH_LOG1P_FN __device__ __forceinline__
#define SH_LOG1P_TAB __device__
#else
#define SH_LOG1P_FN static inline
#define SH_LOG1P_TAB static
#endif

namespace sh {

struct __attribute__((aligned(16))) LogStep {
  float inv;  // 1 / c
  float lo;   // log c, low and high part
  double hi;
};
constexpr int kLogSteps = 128;
SH_LOG1P_TAB const LogStep kLogTable[kLogSteps] = {
    {0x1p+0f, 0x0p+0f, 0x0p+0},
    {0x1.fap-1f, 0x1.455442p-44f, 0x1.82448a388p-7},
    {0x1.f64p-1f, 0x1.59a5e2p-44f, 0x1.3b024b78cp-6},
    {0x1.f24p-1f, 0x1.a3d886p-44f, 0x1.be0422fcdp-6},
    {0x1.ee8p-1f, 0x1.a9cc78p-44f, 0x1.1ce5a62bcp-5},
    {0x1.ebp-1f, -0x1.8888dep-44f, 0x1.5715c4c04p-5},
    {0x1.e74p-1f, -0x1.ba22dp-45f, 0x1.95e430f8dp-5},
    {0x1.e3cp-1f, -0x1.8e40e4p-45f, 0x1.d0f2c1dda8p-5},
    {0x1.ep-1f, -0x1.7e5dd8p-46f, 0x1.08598b59e4p-4},
    {0x1.dccp-1f, 0x1.4b838ap-45f, 0x1.242d6c1a58p-4},
    {0x1.d94p-1f, 0x1.365ac6p-45f, 0x1.425bce8474p-4},
    {0x1.d5cp-1f, 0x1.45cb1p-44f, 0x1.60c38ba798p-4},
    {0x1.d28p-1f, 0x1.3c88c4p-44f, 0x1.7d33687c28p-4},
    {0x1.cf4p-1f, -0x1.a45d04p-46f, 0x1.99d62a65ecp-4},
    {0x1.ccp-1f, 0x1.b1bep-44f, 0x1.b6ac88dad4p-4},
    {0x1.c8cp-1f, 0x1.f9a80ap-44f, 0x1.d3b73f37ep-4},
    {0x1.c58p-1f, 0x1.2e31f6p-44f, 0x1.f0f70cdd98p-4},
    {0x1.c28p-1f, 0x1.630462p-44f, 0x1.06135354d4p-3},
    {0x1.bf4p-1f, -0x1.03dccap-51f, 0x1.14e75b48ap-3},
    {0x1.bc4p-1f, -0x1.a3c2a6p-45f, 0x1.22aff2ddbep-3},
    {0x1.b94p-1f, -0x1.819b9p-45f, 0x1.3090733ce4p-3},
    {0x1.b64p-1f, -0x1.24aa94p-44f, 0x1.3e892fe996p-3},
    {0x1.b38p-1f, 0x1.522edp-46f, 0x1.4b6d6fefe2p-3},
    {0x1.b08p-1f, -0x1.a1d05ap-44f, 0x1.59958ff1d6p-3},
    {0x1.adcp-1f, 0x1.a68934p-44f, 0x1.66a5d42a3ap-3},
    {0x1.abp-1f, -0x1.d66a9p-44f, 0x1.73cb9074fep-3},
    {0x1.a84p-1f, -0x1.ff00cp-44f, 0x1.81070bd7bap-3},
    {0x1.a58p-1f, 0x1.b7d5cap-44f, 0x1.8e588ebac2p-3},
    {0x1.a2cp-1f, -0x1.e2c9fap-46f, 0x1.9bc062f27p-3},
    {0x1.ap-1f, -0x1.872436p-45f, 0x1.a93ed3c8aep-3},
    {0x1.9d8p-1f, 0x1.9b50e8p-44f, 0x1.b5971a213ap-3},
    {0x1.9bp-1f, -0x1.92e0eep-45f, 0x1.c2028ab18p-3},
    {0x1.984p-1f, -0x1.810b32p-46f, 0x1.cfc25714bep-3},
    {0x1.95cp-1f, 0x1.eb37aap-44f, 0x1.dc56cae452p-3},
    {0x1.934p-1f, 0x1.78e13ep-44f, 0x1.e8ff2622bap-3},
    {0x1.90cp-1f, 0x1.41b254p-44f, 0x1.f5bba8306p-3},
    {0x1.8e8p-1f, 0x1.1cd8d6p-44f, 0x1.00a1c6addap-2},
    {0x1.8cp-1f, -0x1.e76324p-44f, 0x1.07138604d6p-2},
    {0x1.898p-1f, 0x1.ee8c88p-46f, 0x1.0d8fb813ebp-2},
    {0x1.874p-1f, -0x1.bd0584p-44f, 0x1.136ef02e83p-2},
    {0x1.85p-1f, 0x1.7d2f74p-45f, 0x1.1956d3b9bcp-2},
    {0x1.82cp-1f, 0x1.6d6d4p-45f, 0x1.1f477c7573p-2},
    {0x1.808p-1f, 0x1.b1d7acp-44f, 0x1.25410494e5p-2},
    {0x1.7e4p-1f, -0x1.e7d8c6p-47f, 0x1.2b4386c169p-2},
    {0x1.7cp-1f, -0x1.8e27aep-45f, 0x1.314f1e1d36p-2},
    {0x1.79cp-1f, 0x1.18b1f2p-44f, 0x1.3763e64645p-2},
    {0x1.778p-1f, -0x1.22c7c2p-45f, 0x1.3d81fb5947p-2},
    {0x1.758p-1f, 0x1.90644p-44f, 0x1.42f9f3ff62p-2},
    {0x1.734p-1f, 0x1.b90566p-44f, 0x1.4929e8db4ep-2},
    {0x1.714p-1f, 0x1.840474p-46f, 0x1.4eb1f36b07p-2},
    {0x1.6f4p-1f, 0x1.258e66p-45f, 0x1.5441aecbc6p-2},
    {0x1.6dp-1f, -0x1.7c79bp-48f, 0x1.5a8cadbbeep-2},
    {0x1.6bp-1f, 0x1.ebe918p-46f, 0x1.602d08af09p-2},
    {0x1.69p-1f, 0x1.544fd2p-51f, 0x1.65d558d4cep-2},
    {0x1.67p-1f, 0x1.fe675p-45f, 0x1.6b85b4cffap-2},
    {0x1.654p-1f, 0x1.0fb168p-44f, 0x1.7086b1162bp-2},
    {0x1.634p-1f, 0x1.b7826ep-44f, 0x1.76466197e3p-2},
    {0x1.614p-1f, -0x1.c64e12p-45f, 0x1.7c0e612786p-2},
    {0x1.5f8p-1f, -0x1.3a3e94p-47f, 0x1.812444990bp-2},
    {0x1.5d8p-1f, 0x1.239fc8p-44f, 0x1.86fc19d051p-2},
    {0x1.5bcp-1f, 0x1.27c2ecp-45f, 0x1.8c1ffe4002p-2},
    {0x1.59cp-1f, 0x1.8d62eep-44f, 0x1.920800ccb9p-2},
    {0x1.58p-1f, 0x1.ab73b2p-44f, 0x1.973a343135p-2},
    {0x1.564p-1f, -0x1.44e114p-46f, 0x1.9c73305d48p-2},
    {0x1.548p-1f, -0x1.2ca6dp-49f, 0x1.a1b3071f76p-2},
    {0x1.52cp-1f, 0x1.58d4a8p-44f, 0x1.a6f9ca8cbcp-2},
    {0x1.51p-1f, 0x1.bc0e8cp-48f, 0x1.ac478d0205p-2},
    {0x1.4f4p-1f, -0x1.2a5adep-47f, 0x1.b19c6125a7p-2},
    {0x1.4d8p-1f, 0x1.8e7e66p-44f, 0x1.b6f859e8efp-2},
    {0x1.4bcp-1f, -0x1.01fe16p-44f, 0x1.bc5b8a89b6p-2},
    {0x1.4a4p-1f, 0x1.7735a6p-44f, 0x1.c0ff81c705p-2},
    {0x1.488p-1f, -0x1.f0b4f8p-52f, 0x1.c6704e4017p-2},
    {0x1.46cp-1f, 0x1.542dp-49f, 0x1.cbe88b44dcp-2},
    {0x1.454p-1f, -0x1.143cfp-45f, 0x1.d09ebaee2ap-2},
    {0x1.43cp-1f, -0x1.86220ap-46f, 0x1.d55a7df2b2p-2},
    {0x1.42p-1f, 0x1.856f4ap-44f, 0x1.dae75484c9p-2},
    {0x1.408p-1f, 0x1.5d4a8p-46f, 0x1.dfaf59de8cp-2},
    {0x1.3fp-1f, 0x1.df865cp-44f, 0x1.e47d1d32e6p-2},
    {0x1.3d4p-1f, 0x1.72cc32p-48f, 0x1.ea1f2acdd5p-2},
    {0x1.3bcp-1f, -0x1.8039c6p-44f, 0x1.eef98ee334p-2},
    {0x1.3a4p-1f, 0x1.5d6d98p-47f, 0x1.f3d9dd82abp-2},
    {0x1.38cp-1f, 0x1.15162ep-46f, 0x1.f8c0252a83p-2},
    {0x1.374p-1f, 0x1.7cada8p-46f, 0x1.fdac748e87p-2},
    {0x1.35cp-1f, -0x1.4240ap-45f, 0x1.014f6d4c878p-1},
    {0x1.348p-1f, 0x1.524198p-45f, 0x1.03617096e08p-1},
    {0x1.33p-1f, -0x1.fcfe7ap-44f, 0x1.05e04c1aa3p-1},
    {0x1.318p-1f, -0x1.8a931ep-46f, 0x1.086248abc5p-1},
    {0x1.3p-1f, -0x1.82de52p-44f, 0x1.0ae76e2d058p-1},
    {0x1.2ecp-1f, -0x1.ce1f0ep-44f, 0x1.0d037d237f8p-1},
    {0x1.2d4p-1f, -0x1.117a8ap-45f, 0x1.0f8e82914p-1},
    {0x1.2cp-1f, 0x1.53cdc2p-44f, 0x1.11af823c758p-1},
    {0x1.2a8p-1f, 0x1.11b7bep-45f, 0x1.1440833addp-1},
    {0x1.294p-1f, 0x1.cad3f4p-44f, 0x1.16668af4ddp-1},
    {0x1.27cp-1f, -0x1.ef50dep-45f, 0x1.18fda3ecf68p-1},
    {0x1.268p-1f, 0x1.3e8a5ep-45f, 0x1.1b28cbb6ec8p-1},
    {0x1.254p-1f, 0x1.8abd0ep-45f, 0x1.1d5650035a8p-1},
    {0x1.24p-1f, -0x1.a7242cp-45f, 0x1.1f8635fc618p-1},
    {0x1.22cp-1f, 0x1.fc6396p-48f, 0x1.21b882dd26p-1},
    {0x1.214p-1f, -0x1.d739dp-44f, 0x1.245e78a85f8p-1},
    {0x1.2p-1f, 0x1.c93c1ep-44f, 0x1.269621134d8p-1},
    {0x1.1ecp-1f, 0x1.d552f2p-46f, 0x1.28d041990bp-1},
    {0x1.1d8p-1f, -0x1.7eadb8p-44f, 0x1.2b0cdfbf7bp-1},
    {0x1.1c4p-1f, 0x1.ccd6dap-44f, 0x1.2d4c011f1dp-1},
    {0x1.1bp-1f, 0x1.bcccfep-44f, 0x1.2f8dab6363p-1},
    {0x1.1ap-1f, -0x1.74e93cp-45f, 0x1.315da443408p-1},
    {0x1.18cp-1f, -0x1.d3141ap-45f, 0x1.33a3ed10da8p-1},
    {0x1.178p-1f, 0x1.cfc32ep-45f, 0x1.35eccf0ac6p-1},
    {0x1.164p-1f, -0x1.3aebc2p-48f, 0x1.383850278dp-1},
    {0x1.15p-1f, 0x1.112e02p-45f, 0x1.3a86767257p-1},
    {0x1.14p-1f, -0x1.2b7368p-47f, 0x1.3c6080c36cp-1},
    {0x1.12cp-1f, -0x1.254ca4p-44f, 0x1.3eb37978b88p-1},
    {0x1.11cp-1f, -0x1.33298cp-44f, 0x1.409167679ep-1},
    {0x1.108p-1f, 0x1.7e040ap-46f, 0x1.42e946de08p-1},
    {0x1.0f4p-1f, 0x1.9411fcp-46f, 0x1.4543e863cp-1},
    {0x1.0e4p-1f, 0x1.56e0d6p-44f, 0x1.472803f35e8p-1},
    {0x1.0d4p-1f, -0x1.c2e48ap-48f, 0x1.490deaf1a4p-1},
    {0x1.0cp-1f, -0x1.f04776p-44f, 0x1.4b6fd6f971p-1},
    {0x1.0bp-1f, 0x1.d0f65ap-44f, 0x1.4d59d43fda8p-1},
    {0x1.09cp-1f, 0x1.0b8f8p-46f, 0x1.4fc0e728a38p-1},
    {0x1.08cp-1f, 0x1.6805ccp-44f, 0x1.51af0c774ap-1},
    {0x1.07cp-1f, 0x1.84ea8ep-44f, 0x1.539f107e1dp-1},
    {0x1.06cp-1f, 0x1.079b0ep-47f, 0x1.5590f6e02f8p-1},
    {0x1.058p-1f, 0x1.a9786ep-44f, 0x1.580202c6c7p-1},
    {0x1.048p-1f, 0x1.47ffa6p-44f, 0x1.59f833f9d4p-1},
    {0x1.038p-1f, 0x1.0e0674p-45f, 0x1.5bf053a4868p-1},
    {0x1.028p-1f, 0x1.a7e8ccp-44f, 0x1.5dea65985ap-1},
    {0x1.018p-1f, 0x1.920e2ap-45f, 0x1.5fe66db2288p-1},
    {0x1.008p-1f, -0x1.cc9ee2p-44f, 0x1.61e46fda568p-1},
};

// 0 <= y < 2^1000; tab: kLogTable or a copy
template <typename Tab>
SH_LOG1P_FN double log1p_table(double y, Tab tab) {
  const double u = 1.0 + y, b = u - 1.0;
  const double lost = (1.0 - (u - b)) + (y - b);  // 1 + y = u + lost exactly
  uint64_t bits;
  __builtin_memcpy(&bits, &u, 8);
  const int k = (int)(bits >> 52) - 1023;
  const uint64_t mb = (bits & 0x000fffffffffffffull) | 0x3ff0000000000000ull;
  double m;
  __builtin_memcpy(&m, &mb, 8);
  const LogStep s = tab[(bits >> 45) & 127];
  const double inv = s.inv;
  const double r0 = __builtin_fma(m, inv, -1.0);
  const double d = __builtin_ldexp(lost, -k) * inv, r = r0 + d;
  double p = __builtin_fma(r, -1.0 / 8, 1.0 / 7);
  p = __builtin_fma(p, r, -1.0 / 6);
  p = __builtin_fma(p, r, 1.0 / 5);
  p = __builtin_fma(p, r, -1.0 / 4);
  p = __builtin_fma(p, r, 1.0 / 3);
  p = __builtin_fma(p, r, -1.0 / 2);
  const double kd = (double)k;
  const double low = __builtin_fma(kd, 0x1.ef35793c7673p-45, (double)s.lo);
  const double high = __builtin_fma(kd, 0x1.62e42fefa38p-1, s.hi);
  const double sum = high + r0;
  const double rest = ((high - sum) + r0) + d;  // high is 0 or larger than r0
  return sum + (rest + __builtin_fma(p, r * r, low));
}

}  // namespace sh
