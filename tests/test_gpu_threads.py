"""Host threads: tq_linear_forward on different layers from several threads at once (each thread its own
stream and buffers), and on ONE layer from several threads for the paths that use no per-layer workspace
(one row per call).  Results must equal the single-threaded ones bit for bit; tq_last_error is per thread."""
import ctypes
import threading

import numpy as np
import pytest

from test_gpu_graph import _Hip, _bits, _layer

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tq():
    import __graft_entry__ as entry
    pkg = entry.load_package()
    pkg.lib()
    return pkg


def test_forward_from_four_threads(tq, oracle):
    o = oracle
    shapes = [(384, 1024, 512, "shared"), (200, 2048, 256, "dual"), (96, 5120, 512, "shared"), (130, 1536, 512, "primary_only")]
    layers = [_layer(tq, o, out, inf, bs, mode, seed=20 + i)[0] for i, (out, inf, bs, mode) in enumerate(shapes)]
    shared_layer = layers[0]
    rng = np.random.default_rng(9)
    xb = [{b: _bits(o, rng, b, inf) for b in (1, 4)} for (_, inf, _, _) in shapes]
    hips = [_Hip() for _ in shapes]
    # single-threaded results first
    want, xs, ys = [], [], []
    for i, (out, inf, bs, mode) in enumerate(shapes):
        h = hips[i]
        layers[i].reserve(4)
        xs.append({b: h.upload(xb[i][b]) for b in (1, 4)})
        ys.append({b: h.alloc(b * out * 4) for b in (1, 4)})
        w = {}
        for b in (1, 4):
            layers[i].forward_device(xs[i][b], tq.BF16, b, ys[i][b], tq.F32, h.stream)
            w[b] = h.download(ys[i][b], (b, out))
        want.append(w)
    y_shared = [h.alloc(shapes[0][0] * 4) for h in hips]
    failures = []

    def work(i):
        try:
            h, (out, inf, bs, mode) = hips[i], shapes[i]
            for turn in range(40):
                b = (1, 4)[turn % 2]
                layers[i].forward_device(xs[i][b], tq.BF16, b, ys[i][b], tq.F32, h.stream)
                # one row of the layer every thread shares: no per-layer workspace involved
                shared_layer.forward_device(xs[0][1], tq.BF16, 1, y_shared[i], tq.F32, h.stream)
                if turn % 10 == 9:
                    assert h.rt.hipStreamSynchronize(h.stream) == 0
                    got = np.empty((b, out), np.float32)
                    assert h.rt.hipMemcpy(got.ctypes.data_as(ctypes.c_void_p), ys[i][b], got.nbytes, 2) == 0
                    if not np.array_equal(got, want[i][b]):
                        failures.append((i, turn, "own layer"))
                    got = np.empty((1, shapes[0][0]), np.float32)
                    assert h.rt.hipMemcpy(got.ctypes.data_as(ctypes.c_void_p), y_shared[i], got.nbytes, 2) == 0
                    if not np.array_equal(got, want[0][1]):
                        failures.append((i, turn, "shared layer"))
            # an error in this thread is this thread's message
            rc = tq.lib().tq_linear_forward(layers[i]._h, None, tq.BF16, 1, ys[i][1], tq.F32, None)
            if rc == 0 or "NULL" not in tq.last_error():
                failures.append((i, "error message", tq.last_error()))
        except Exception as e:                                 # noqa: BLE001 - reported through the list
            failures.append((i, repr(e)))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(shapes))]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=100)
    assert not any(t.is_alive() for t in threads)
    assert not failures, failures
    for layer in layers:
        layer.close()
    for h in hips:
        h.close()


def test_conversions_from_threads_share_kept_memory(tq, oracle):
    """Fit and quantization of layers of different sizes from three threads at once, with the kept device memory given
    back now and then: what a call returns is what it returns alone (a first call on fresh memory, checked against the
    oracle), whatever the block held before."""
    rng = np.random.default_rng(12)
    weights = [(rng.standard_normal(s) * 0.02).astype(np.float32) for s in ((1030, 1024), (515, 2048), (4099, 1024))]
    tq.lib().tq_quantizer_release_workspaces()

    def convert(w):
        p, r = tq.fit_layer_codebooks(w, 512)
        q = tq.quantize_weight(w, p, r, 4, 4, 512, False)
        return [p.centroids, r.centroids, q.packed_primary, q.packed_residual, q.norms, q.seeds], p, r

    want = [convert(w)[0] for w in weights]
    _, p, r = convert(weights[0])
    ref = oracle.quantize_weight(weights[0], p, r, 4, 4, 512, False)
    assert np.array_equal(ref.packed_primary, want[0][2])
    failures = []

    def work(i):
        try:
            for turn in range(8):
                k = (i + turn) % len(weights)
                got = convert(weights[k])[0]
                if not all(np.array_equal(np.asarray(a), np.asarray(b)) for a, b in zip(got, want[k])):
                    failures.append((i, turn, k))
                if turn % 4 == i:
                    tq.lib().tq_quantizer_release_workspaces()
        except Exception as e:                                  # noqa: BLE001
            failures.append((i, repr(e)))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    tq.lib().tq_quantizer_release_workspaces()
    assert not failures, failures
