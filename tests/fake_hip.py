"""The kernels that contexts launch, on a HIP runtime without a device
(fake_hip.cpp), each context in a process of its own request: launches()."""
import ctypes
import json
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


def build(folder):
    so = os.path.join(str(folder), "fake_hip.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-o", so, os.path.join(HERE, "fake_hip.cpp")],
                   check=True)
    return so


def launches(so, contexts, cus=256, env=None):
    """Kernel names (template arguments included) of the third of three steps of
    each context, a list of (sizes, precision, options)."""
    e = dict(os.environ, FAKE_HIP_CUS=str(cus), **(env or {}))
    r = subprocess.run([sys.executable, os.path.abspath(__file__), so, json.dumps(contexts)], env=e, check=True,
                       capture_output=True, text=True, timeout=300)
    return json.loads(r.stdout.splitlines()[-1])


def main(so, contexts):
    fake = ctypes.CDLL(so, mode=ctypes.RTLD_GLOBAL)
    fake.fake_hip_launches.restype = ctypes.c_char_p
    sys.path.insert(0, os.path.join(ROOT, "ek-pnp_amd"))
    import ekpnp

    out = []
    for sizes, precision, options in contexts:
        s = ekpnp.Solver([ekpnp.lattice_params(nx, ny, kappa_h=min(4.0, 0.15 * ny)) for nx, ny in sizes],
                         precision=precision, use_graph=False, **options)
        s.initialization(ekpnp.COLD_NOISE, 0)
        s.init_equilibrium()
        s.step(1)  # from the pre-collision form
        fake.fake_hip_launches()
        s.step(3)
        out.append([line.rsplit(" ", 1)[0] for line in fake.fake_hip_launches().decode().splitlines()])
        s.close()
    print(json.dumps(out))


if __name__ == "__main__":
    main(sys.argv[1], json.loads(sys.argv[2]))
