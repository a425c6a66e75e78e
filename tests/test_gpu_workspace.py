"""lkhip_matmul's kept workspaces: products that share them equal the same
products alone."""
import ctypes as C
import threading

import numpy as np
import pytest

import oracle
from lokal_amd import kernels as K
from lokal_amd import synth

pytestmark = pytest.mark.gpu


def test_matmul_workspace_is_shared_in_stream_order():
    """Products of several sizes, back to back on the null stream and on two
    created streams, use kept workspaces: each equals the same product alone,
    also after a stream and every weight are gone."""
    rng = np.random.default_rng(5)
    shapes = [(2048, 2048, 100), (4864, 896, 64), (1024, 4864, 200), (6000, 896, 512)]
    for _ in range(2):
        ws, xs, alone = [], [], []
        for rows, cols, n in shapes:
            ws.append(K.Weight(synth.Q8_0, rows, cols, synth.gen_weight(synth.Q8_0, 3, f"{rows}", rows, cols).data))
            xs.append(K.DeviceArray.from_numpy(rng.standard_normal((n, cols)).astype(np.float32)))
            y = K.DeviceArray((n, rows))
            K.matmul(ws[-1], xs[-1], n, y)
            alone.append(y.numpy())
        streams = [K.Stream(), K.Stream()]
        outs = []
        for rep in range(3):
            for st in (None, *streams):
                for w, x, (rows, cols, n) in zip(ws, xs, shapes):
                    y = K.DeviceArray((n, rows))
                    K.matmul(w, x, n, y, stream=st.ptr if st else None)
                    outs.append(y)
        K.synchronize()
        for i, y in enumerate(outs):
            assert np.array_equal(y.numpy(), alone[i % len(shapes)]), i
        for st in streams:
            st.close()
        for w in ws:
            w.close()


def test_matmul_workspace_from_several_threads():
    """Two threads on streams of their own and two on the null stream, products of
    several sizes at once: each equals the same product alone.  A fifth makes and
    destroys streams meanwhile."""
    rng = np.random.default_rng(6)
    cases = []
    for rows, cols, n in [(2048, 2048, 100), (4864, 896, 64), (1024, 4864, 200)]:
        w = K.Weight(synth.Q8_0, rows, cols, synth.gen_weight(synth.Q8_0, 3, f"{rows}", rows, cols).data)
        x, y = K.DeviceArray.from_numpy(rng.standard_normal((n, cols)).astype(np.float32)), K.DeviceArray((n, rows))
        K.matmul(w, x, n, y)
        cases.append((w, x, n, y.numpy()))
    bad = []

    def work(k, st):
        try:
            for rep in range(12):
                w, x, n, want = cases[(k + rep) % len(cases)]
                y = K.DeviceArray(want.shape)
                K.matmul(w, x, n, y, stream=st.ptr if st else None)
                if not np.array_equal(y.numpy(), want):
                    bad.append((k, rep))
        except Exception as e:  # noqa: BLE001 -- told by the main thread
            bad.append((k, e))

    def come_and_go():
        w, x, n, want = cases[0]
        for _ in range(6):
            st, y = K.Stream(), K.DeviceArray(want.shape)
            K.matmul(w, x, n, y, stream=st.ptr)
            st.synchronize()
            if not np.array_equal(y.numpy(), want):
                bad.append("come_and_go")
            st.close()

    streams = [K.Stream(), K.Stream(), None, None]
    threads = [threading.Thread(target=work, args=(k, s)) for k, s in enumerate(streams)]
    threads.append(threading.Thread(target=come_and_go))
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
    for s in streams[:2]:
        s.close()


@pytest.mark.parametrize("rows,cols,n,memory", [(4864, 896, 512, False), (2048, 2048, 100, True)])
def test_matmul_under_capture(rows, cols, n, memory):
    """A product that needs no partial sums records kernels only, so its graph can
    be instantiated twice; one that splits K allocates inside the graph.  Replays
    on new rows, eager products between them, equal the eager result within the
    rounding of two f32 sums of K products, (K / 32 + 40) * 2^-24 of the |terms| each."""
    hip = C.CDLL("libamdhip64.so")
    rng = np.random.default_rng(n)
    data = synth.gen_weight(synth.Q8_0, 3, "w", rows, cols).data
    w = K.Weight(synth.Q8_0, rows, cols, data)
    ref = np.abs(oracle.dequant_row(synth.Q8_0, data, rows * cols).reshape(rows, cols))
    x, y, eager = K.DeviceArray((n, cols)), K.DeviceArray((n, rows)), K.DeviceArray((n, rows))
    x.zero()
    st, graph, num = K.Stream(), C.c_void_p(), C.c_size_t()
    K.matmul(w, x, n, y, stream=st.ptr)
    st.synchronize()
    assert hip.hipStreamBeginCapture(st.ptr, 0) == 0
    K.matmul(w, x, n, y, stream=st.ptr)
    assert hip.hipStreamEndCapture(st.ptr, C.byref(graph)) == 0
    assert hip.hipGraphGetNodes(graph, None, C.byref(num)) == 0
    nodes, kind, kinds = (C.c_void_p * num.value)(), C.c_int(), []
    assert hip.hipGraphGetNodes(graph, nodes, C.byref(num)) == 0
    for node in nodes:
        assert hip.hipGraphNodeGetType(C.c_void_p(node), C.byref(kind)) == 0
        kinds.append(kind.value)
    assert (set(kinds) != {0}) == memory  # 0: kernels
    execs = [C.c_void_p() for _ in range(1 if memory else 2)]
    for ex in execs:
        assert hip.hipGraphInstantiate(C.byref(ex), graph, None, None, C.c_size_t(0)) == 0
    for rep in range(4):
        xv = rng.standard_normal((n, cols)).astype(np.float32)
        x.upload(xv)
        K.matmul(w, x, n, eager)
        K.synchronize()
        y.zero()
        K.synchronize()
        assert hip.hipGraphLaunch(execs[rep % len(execs)], st.ptr) == 0
        st.synchronize()
        bar = 2 * (cols / 32 + 40) * 2.0 ** -24 * (np.abs(xv) @ ref.T)
        assert np.all(np.abs(y.numpy() - eager.numpy()) <= bar)
    for ex in execs:
        assert hip.hipGraphExecDestroy(ex) == 0
    assert hip.hipGraphDestroy(graph) == 0
    st.close()
