"""The host calls' pinned memory: from an engine's first host call on.

An engine that only the device entry points use pins nothing.  Small ones share
64 + 16 blocks of the process, larger ones and those beyond map 16 bytes a parameter
of their own.
"""

from __future__ import annotations

import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _mapped_bytes():
    with open("/proc/self/status") as f:
        return 1024 * next(int(line.split()[1]) for line in f if line.startswith("VmSize:"))


def test_the_first_host_call_maps_a_large_block(backend_module):
    n, layers = 2, 1 << 18
    p = np.zeros(2 * n * layers)
    warm = backend_module.RingIsingCudaBackend(n, 4, 1.0, "structured_adjoint", 8, False)
    warm.energy_and_grad(p[:16])
    eng = backend_module.RingIsingCudaBackend(n, layers, 1.0, "structured_adjoint", 8, False)
    before = _mapped_bytes()
    eng.energy_and_grad(p, False)
    assert _mapped_bytes() - before >= 16 * p.size


def test_engines_share_the_blocks(oracle, backend_module):
    # more engines than blocks, all alive, called in turn; then threads that make,
    # call and drop them
    n, layers = 5, 2
    rng = np.random.default_rng(62)
    params = [rng.uniform(0, 2 * np.pi, 2 * n * layers) for _ in range(90)]
    refs = [oracle.energy_and_grad(n, layers, 1.0, p.reshape(layers, n, 2)) for p in params]

    def make():
        return backend_module.RingIsingCudaBackend(n, layers, 1.0, "structured_adjoint", 8, False)

    def check(eng, k):
        out = eng.energy_and_grad(params[k])
        assert abs(out["energy"] - refs[k][0]) <= 1e-10
        assert np.max(np.abs(np.asarray(out["gradient"]) - np.ravel(refs[k][1]))) <= 1e-10

    print("case 90 engines", flush=True)
    engines = [make() for _ in params]
    for _ in range(2):
        for k, eng in enumerate(engines):
            check(eng, k)
    del engines[::2]
    for k, eng in enumerate(engines):
        check(eng, k)
    errors = []

    def work(first):
        try:
            for k in range(first, 90, 4):
                check(make(), k)
        except Exception as error:
            errors.append(error)

    threads = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors[0]
