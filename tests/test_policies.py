"""The library's kernels with a caller's policies, of the shapes that the
reference's functors have and nothing more (no GPU: it has to compile)."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "miniaero_amd", "csrc")

POLICIES = """
struct MyFlux {  // Roe_Flux.h:50-54
  template <class T>
  MA_HD void compute_flux(const T* V_L, const T* V_R, T* F, const T* n, const T* t, const T* b) const {
    for (int k = 0; k < 5; ++k) F[k] = T(0.5) * (V_L[k] + V_R[k]) * (n[0] + t[1] + b[2]);
  }
};
struct MyViscousFlux {  // Viscous_Flux.h:39-99
  enum { isViscous = true };
  double prandtl;
  template <class T>
  MA_HD void compute_flux(const T g[5][3], const T* V, const T* a, T* F) const {
    for (int k = 0; k < 5; ++k) F[k] = T(1e-5) * V[4] * (g[k][0] * a[0] + g[k][1] * a[1] + g[k][2] * a[2]);
  }
};
struct MyLimiter {  // VenkatLimiter.h:45
  template <class T>
  static MA_HD T limit(T dumax, T dumin, T du, T deltax3) {
    return du > T(0) ? smin(T(1), dumax / du) : du < T(0) ? smin(T(1), dumin / du) : T(1) + T(0) * deltax3;
  }
};
struct MyInflowBC {  // Inflow_BC.h:61-73
  template <class T, class Inv, class Wall>
  MA_HD void operator()(const T* V, const FaceFrameT<T>& face, const double* inflow, T wall_inv, const Inv& inv,
                        const Wall&, T* out) const {
    T vr[5], F[5];
    for (int k = 0; k < 5; ++k) vr[k] = T(0.5) * (V[k] + T(inflow[k])) + T(0) * wall_inv;
    inviscid_flux(inv, V, vr, F, face);
    for (int k = 0; k < 5; ++k) out[k] = -F[k];
  }
};
struct MyBoundaries : ReferenceBoundaries {
  using Inflow = MyInflowBC;
};
"""

EDITS = {
    "flux": [("using Inviscid = ma::RoeFlux;", "using Inviscid = ma::MyFlux;")],
    "viscous flux": [("lim<true, ma::NewtonianViscousFlux, T>", "lim<true, ma::MyViscousFlux, T>"),
                     ("lim<false, ma::NewtonianViscousFlux, T>", "lim<false, ma::MyViscousFlux, T>"),
                     ("paired_limiter<ma::NewtonianViscousFlux>", "paired_limiter<ma::MyViscousFlux>")],
    "limiter": [("ma::VenkatLimiter", "ma::MyLimiter")],
    "boundaries": [("using Boundaries = ma::ReferenceBoundaries;", "using Boundaries = ma::MyBoundaries;")],
}

CHECK = """
namespace {
static_assert(ma::pair_policies<ma::NewtonianViscousFlux, ma::VanAlbadaLimiter, ma::ReferenceBoundaries>, "");
static_assert(ma::pair_policies<ma::NoViscousFlux, ma::VenkatLimiter, ma::ReferenceBoundaries>, "");
static_assert(!ma::pair_policies<ma::MyViscousFlux, ma::VenkatLimiter, ma::ReferenceBoundaries>, "");
static_assert(!ma::pair_policies<ma::NoViscousFlux, ma::MyLimiter, ma::ReferenceBoundaries>, "");
static_assert(!ma::pair_policies<ma::NoViscousFlux, ma::VenkatLimiter, ma::MyBoundaries>, "");
}
"""


@pytest.mark.parametrize("what", sorted(EDITS))
def test_documented_policy_shapes_compile(tmp_path, what):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    src = tmp_path / "miniaero_amd" / "csrc"
    shutil.copytree(CSRC, src)
    shutil.copytree(os.path.join(CSRC, "..", "..", "include"), tmp_path / "include")
    text = (src / "physics.hpp").read_text()
    at = text.rindex("}  // namespace ma")
    (src / "physics.hpp").write_text(text[:at] + POLICIES + text[at:])
    text = (src / "solver.hip").read_text()
    for old, new in EDITS[what]:
        assert old in text
        text = text.replace(old, new)
    (src / "solver.hip").write_text(text + CHECK)
    r = subprocess.run([hipcc, "-fsyntax-only", "-std=c++17", "-ffp-contract=off", "-fno-fast-math",
                        "--offload-arch=gfx950", "--offload-device-only", str(src / "solver.hip")],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-3000:]
