"""The server's worker thread does not hold a core while a long batch is on the device: past a
millisecond of looking for its end without a pause it waits."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_long_batches_do_not_hold_a_core():
    import eig_amd
    N, M, K, batch, reps = 64, 6000000, 16, 1024, 8
    rng = np.random.default_rng(3)
    eng = eig_amd.Engine(0)
    pool = None
    try:
        thr = (rng.uniform(0.1, 0.9, (2, M)) * 2.0 ** 32).astype(np.uint32)
        anc = np.repeat((np.arange(N) % 2).astype(np.int32)[:, None], 3, axis=1)
        eng.synth(M, N, thr, anc, np.full((N, 2), 0xFFFFFFFF, np.uint32), 0, 7)
        eng.select(np.arange(N, dtype=np.int32))
        eng.snpstats(fetch=False)
        vec = np.linalg.qr(rng.standard_normal((N, K)))[0].T
        eng.loadings(np.ascontiguousarray(vec), want_ffvecs=False)
        with eig_amd.Server(eng, nlanes=1, max_batch=batch) as srv:
            pool = eng.dev_alloc(batch * srv.rowpad)  # any bytes are valid rows
            print("[gpu-case] server worker, long batches", flush=True)
            go = lambda: [srv.submit(device_ptr=pool, nq=batch, stride=srv.rowpad) for _ in range(reps)]
            for t in go():
                srv.poll(t)
            w0, c0 = time.perf_counter(), time.process_time()
            for t in go():
                srv.poll(t)
            wall, cpu = time.perf_counter() - w0, time.process_time() - c0
    finally:
        if pool is not None:
            eng.dev_free(pool)
        eng.close()
    print(f"wall {1e3 * wall:.1f} ms, CPU {1e3 * cpu:.1f} ms")
    # a batch is several times the millisecond: a worker that never paused would use it all
    assert wall / reps > 4e-3
    assert cpu < 0.6 * wall
