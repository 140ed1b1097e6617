"""Solves of several threads on one GPU: each takes the path, and gives the
bits, that it takes and gives alone."""

import threading

import pytest
import torch

from test_gpu_persist import model_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_results_do_not_depend_on_other_threads(precision):
    sizes = [(8, 8, 8), (7, 9, 8), (15, 14, 16), (3, 2, 4)]

    def solve(m):
        u = m.solve(precision=precision, preconditioner="block_jacobi", stol=1e-10)[0]
        return u.detach(), m.last_solve_info["forward"]["pcg"][0]["path"]

    models = [model_of("hexa1", n) for n in sizes]
    want = [solve(m)[0] for m in models]
    torch.cuda.synchronize()
    start = threading.Barrier(len(models))
    errors = []

    def work(k):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                start.wait()
                for i in range(20):
                    u, path = solve(models[k])
                    torch.cuda.current_stream().synchronize()
                    if path != "persistent" or not torch.equal(u, want[k]):
                        errors.append((k, i, path))
        except Exception as e:  # noqa: BLE001 - reported by the assertion
            errors.append(repr(e))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(models))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors
