"""How the library would run a convolution, asked on the CPU: a small program
(tests/routes/routes.cpp) linked against the static archive prints a problem's
transform lengths, whether it takes the whole-plane kernels, and its
workspace."""
import os
import subprocess

import pytest

from test_gpu_planes import REGULAR_PLANES, WIDE_PLANES

ROOT = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..")
MODES = {"periodic": 0, "zero": 1, "nearest": 2, "reflect": 3, "mirror": 4}


@pytest.fixture(scope="session")
def routes(fc, tmp_path_factory):
    """routes([(nx, ny, nz, kx, ky, kz, boundary), ...]) -> [(px, py, pz,
    plane forward, plane inverse, workspace bytes), ...]"""
    prog = str(tmp_path_factory.mktemp("routes") / "routes")
    csrc = fc._lib.CSRC
    archive = os.path.join(os.path.dirname(fc._lib.LIB_PATH),
                           "libFourierConvolutionCUDALib_static.a")
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I", csrc,
                    "-I/opt/rocm/include", os.path.join(ROOT, "tests", "routes", "routes.cpp"),
                    archive, "-L/opt/rocm/lib", "-lamdhip64", "-Wl,-rpath,/opt/rocm/lib",
                    "-lpthread", "-o", prog], check=True)

    def ask(problems):
        # every split form on, so that no rule asks a device for its CU count
        env = dict(os.environ, FCAMD_PLANE_SPLIT="1")
        env.pop("FCAMD_NO_PLANES", None)
        env.pop("FCAMD_NO_STATIC", None)
        r = subprocess.run([prog], input="\n".join(" ".join(map(str, p)) for p in problems),
                           env=env, capture_output=True, text=True)
        assert r.returncode == 0, r.stderr
        out = [tuple(int(v) for v in line.split()) for line in r.stdout.splitlines()]
        assert len(out) == len(problems)
        return out

    return ask


def test_extended_planes_take_no_plane_kernel(routes):
    """Every plane extent with whole-plane kernels, in every boundary mode: a
    transform longer than the plane in x or y has no such kernel (they run the
    image's own plane as a circular one); a plane of its own extents has."""
    planes = REGULAR_PLANES + WIDE_PLANES
    problems = [(nx, ny, 64, kx, ky, kz, b) for nx, ny in planes
                for kx, ky, kz in ((9, 9, 9), (3, 1, 1), (1, 3, 1), (1, 1, 9), (1, 1, 1))
                for b in MODES.values()]
    extended = plain = 0
    for p, (px, py, _, fwd, inv, _) in zip(problems, routes(problems)):
        if (px, py) != p[:2]:
            assert (fwd, inv) == (0, 0), p
            extended += 1
        else:
            assert fwd or inv, p
            plain += 1
    # longer in x or y: 3 kernels x 4 modes of every plane
    assert extended == 12 * len(planes) and plain == 13 * len(planes)
