"""The server at the sizes where its kernels change: one row tile streamed (up to 16
samples), then blocks of one, two and more row tiles a wave, with a last partial stage of
SNPs.  Every sample's result is the same bits as alone, and satisfies its normal equations
(oracle-independent: formed in extended precision from the loadings) to their rounding."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K", [(33, 1), (127, 2), (700, 5), (1025, 11), (4100, 16)])
def test_server_batch_sizes(M, K):
    import eig_amd
    rng = np.random.default_rng(M + K)
    N = 60
    p = rng.uniform(0.05, 0.5, M)
    g = rng.binomial(2, p[:, None], size=(M, N)).astype(np.int32)
    eng = eig_amd.Engine(0)
    try:
        eng.load_packed(O.pack_genotypes(g), N)
        eng.select(np.arange(N, dtype=np.int32))
        st = eng.snpstats()
        vec = np.linalg.qr(rng.standard_normal((N, K)))[0].T
        ff, fx = eng.loadings(np.ascontiguousarray(vec))
        nq = 300
        q = rng.binomial(2, p, size=(nq, M)).astype(np.int32)
        q[rng.random((nq, M)) < 0.3] = 3
        q[5] = 3  # nothing observed
        from eig_amd import synth
        rows = synth.pack_samples(q)
        L = np.longdouble
        e = (fx[:, None] * ff).astype(L)
        keep = st["status"] == 0
        with eig_amd.Server(eng, nlanes=2) as srv:
            alone = []
            for i in range(nq):
                alone.append(srv.poll(srv.submit(rows[i:i + 1])))
            for n in (2, 15, 16, 17, 63, 64, 65, 128, 129, 192, 193, 256, 257, nq):
                print(f"[gpu-case] server M={M} K={K} batch {n}", flush=True)
                co, stt, _ = srv.poll(srv.submit(rows[:n]))
                solo = np.concatenate([a[0] for a in alone[:n]])
                s1 = np.concatenate([a[1] for a in alone[:n]])
                assert np.array_equal(stt, s1)
                assert np.array_equal(co[stt != 2], solo[stt != 2])
            for i in range(0, nq, 37):
                obs = (q[i] != 3) & keep
                co, stt, _ = alone[i]
                assert (stt[0] == 1) == (obs.sum() <= K)
                if stt[0] != 0:
                    continue
                x = (q[i] * st["fancy"].astype(L) - st["mean"].astype(L) * st["fancy"])[obs]
                eo = e[:, obs]
                G, r = eo @ eo.T, eo @ x
                # grids of 2^-53 of the largest entry and a Cholesky backward error
                eps = 2.0 ** -53
                gn = float(np.abs(G).max())
                qg = eps * float(np.abs(e).max()) ** 2
                qr = eps * float((np.abs(e) * st["fancy"] * 3 * (1 + st["mean"])).max())
                tol = K * (M * qg / 2 + 8 * K * K * eps * gn) * np.abs(co[0]).max() + \
                    9 * M * qr / 2 + 16 * eps * np.abs(eo) @ np.abs(x)
                assert np.all(np.abs(G @ co[0].astype(L) - r) <= tol)
    finally:
        eng.close()
