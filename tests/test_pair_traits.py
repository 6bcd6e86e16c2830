"""The functor contract's optional traits (include/xnb_compute_pair.h), checked by the compiler: a
functor that does not say otherwise finds the particle types staged, batched or not."""
import os
import subprocess

from exanbody_amd.build import ARCH, HIPCC

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = """
#include "exanbody_amd/csrc/xnb_pair.h"
namespace xnb {
struct BatchedByType {
  template <int U, bool ENERGY>
  __device__ void batch(const double4& ra, const NbhBatch<U>& nb, double& fx, double&, double&, double&) const {
    for (int u = 0; u < U; u++) fx += nb.type_of(u) * (nb(u).x - ra.x);
  }
};
template <>
struct ComputePairTraits<BatchedByType> {
  static constexpr bool ComputeBufferCompatible = true, BufferLessCompatible = false, CentralType = true, CentralEnergy = false,
                        Batched = true;
};
static_assert(PairTypes<ComputePairTraits<BatchedByType>>::value, "");
static_assert(PairTypes<ComputePairTraits<GravitationalForceFunctor>>::value, "");
static_assert(PairTypes<ComputePairTraits<int>>::value, "");
static_assert(!PairTypes<ComputePairTraits<LennardJonesForceFunctor<true>>>::value, "");
static_assert(!PairTypes<ComputePairTraits<LennardJonesForceFunctor<false>>>::value, "");
}
"""


def test_types_are_staged_unless_the_traits_say_otherwise(tmp_path):
    src = tmp_path / "traits.hip"
    src.write_text(SOURCE)
    r = subprocess.run([HIPCC, f"--offload-arch={ARCH}", "-std=c++17", "-fsyntax-only", f"-I{ROOT}", str(src)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
