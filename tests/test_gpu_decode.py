"""Greedy transducer decode on the device (pkx_transducer_greedy) against the
oracle's restatement of the per-item loops (tdt.cpp / the RNNT loop, which
transducer_batch.cpp reproduces in lockstep).  Bar: identical token ids,
frames and spans per item (the argmax decisions), confidence within 1e-5.
The joint's output weights are scaled up so that the decisions have margins
far above f32 rounding (the device sums the products in another order)."""
import ctypes as C
import threading

import numpy as np
import pytest

import oracle
import pk_model as pm

pytestmark = pytest.mark.gpu


def _model(durations, seed=7, qtype="f32"):
    cfg = pm.Config(d_model=128, n_layers=1, n_heads=2, ff_dim=256, n_mels=64, sub_channels=16, vocab_size=40,
                    joint_hidden=128, pred_hidden=64, pred_rnn_layers=2, tdt_durations=tuple(durations))
    m = pm.add_prediction(pm.synthesize(cfg, qtype, heads=True, seed=seed), seed=seed)
    for n in ("joint.joint_net.2.weight", "joint.joint_net.2.bias"):
        t = m.tensors[n]
        m.tensors[n] = pm.Tensor(t.gtype, t.shape, (t.data * 60.0).astype(np.float32))
    return cfg, m


@pytest.mark.parametrize("kind,max_symbols,qtype", [("tdt", 10, "f32"), ("tdt", 2, "f32"), ("rnnt", 10, "f32"),
                                                     ("rnnt", 1, "f32"), ("tdt", 10, "q8_0")])
def test_greedy_decode_matches_oracle(gpu, stream, kind, max_symbols, qtype):
    durations = (0, 1, 2, 3, 4) if kind == "tdt" else ()
    cfg, m = _model(durations, qtype=qtype)
    gm = gpu.Model.from_tensors(m)
    tr = oracle.Transducer(m)
    rng = np.random.default_rng(11)
    T_valid = [60, 1, 37, 0, 59, 12]
    B, T_max = len(T_valid), 60
    enc = rng.standard_normal((B, T_max, cfg.d_model)).astype(np.float32)
    print(f"[decode] {kind} max_symbols={max_symbols} T={T_valid}", flush=True)
    d_enc = gpu.DeviceArray.from_numpy(enc, stream)
    got = gm.transducer_greedy(d_enc, T_valid, durations=durations, max_symbols=max_symbols, stream=stream)
    total = 0
    for b in range(B):
        ids, fr, cf, sp = tr.greedy(enc[b, :T_valid[b]], durations=durations, max_symbols=max_symbols)
        g_ids, g_fr, g_cf, g_sp = got[b]
        total += len(ids)
        assert np.array_equal(g_ids, ids), (b, g_ids[:20], ids[:20])
        assert np.array_equal(g_fr, fr) and np.array_equal(g_sp, sp)
        assert np.max(np.abs(g_cf - cf), initial=0.0) <= 1e-5
        assert np.all(ids < cfg.vocab_size)
    print(f"[decode] {total} tokens identical", flush=True)
    assert total > 20
    d_enc.free()


@pytest.mark.parametrize("H,Hj,layers,vocab,B", [(20, 36, 1, 30, 1), (36, 20, 3, 43, 16), (340, 1300, 2, 2100, 33)])
def test_greedy_decode_operand_remainders(gpu, stream, H, Hj, layers, vocab, B):
    """Sizes that are no multiple of the products' 16-row tiles and 16-column
    chunks, waves with no chunk and with the most (Hj above 1280), a vocabulary
    of several argmax passes, full and started blocks of 16 items; twice, so that
    the second call finds the first one's workspace."""
    durations = (0, 1, 2)
    cfg = pm.Config(d_model=64, n_layers=1, n_heads=2, ff_dim=128, n_mels=64, sub_channels=16, vocab_size=vocab,
                    joint_hidden=Hj, pred_hidden=H, pred_rnn_layers=layers, tdt_durations=durations)
    m = pm.add_prediction(pm.synthesize(cfg, "f32", heads=True, seed=H), seed=H)
    for n in ("joint.joint_net.2.weight", "joint.joint_net.2.bias"):
        t = m.tensors[n]
        m.tensors[n] = pm.Tensor(t.gtype, t.shape, (t.data * 60.0).astype(np.float32))
    gm = gpu.Model.from_tensors(m)
    tr = oracle.Transducer(m)
    rng = np.random.default_rng(B)
    T_valid = [12] + [int(t) for t in rng.integers(0, 13, B - 1)]
    enc = rng.standard_normal((B, 12, cfg.d_model)).astype(np.float32)
    print(f"[decode] H={H} Hj={Hj} layers={layers} T={T_valid}", flush=True)
    d_enc = gpu.DeviceArray.from_numpy(enc, stream)
    want = [tr.greedy(enc[b, :T_valid[b]], durations=durations, max_symbols=3) for b in range(B)]
    for _ in range(2):
        got = gm.transducer_greedy(d_enc, T_valid, durations=durations, max_symbols=3, stream=stream)
        for b in range(B):
            for i in (0, 1, 3):
                assert np.array_equal(got[b][i], want[b][i]), (b, i, got[b][i], want[b][i])
            # logits below about 1e3, an f32 ulp 6e-5: two ulps move the confidence by at most 2 max|dl| p
            assert np.max(np.abs(got[b][2] - want[b][2]), initial=0.0) <= 2.5e-4
    assert sum(len(w[0]) for w in want) > 0
    d_enc.free()


def test_decode_rejects_bad_arguments(gpu, stream):
    cfg, m = _model((0, 1, 2, 3, 4))
    gm = gpu.Model.from_tensors(m)
    enc = np.zeros((1, 4, cfg.d_model), np.float32)
    d_enc = gpu.DeviceArray.from_numpy(enc, stream)
    with pytest.raises(gpu.PkxError, match="durations"):
        gm.transducer_greedy(d_enc, [4], durations=(0, 1), stream=stream)
    with pytest.raises(gpu.PkxError, match="T_valid"):
        gm.transducer_greedy(d_enc, [5], durations=(0, 1, 2, 3, 4), stream=stream)
    d_enc.free()


def test_greedy_decode_more_items_than_one_pass(gpu, stream):
    """21 items: the matvec kernels take the items in passes of 16 through LDS
    (the second pass reuses the weight rows the wave holds in registers)."""
    durations = (0, 1, 2, 3, 4)
    cfg, m = _model(durations, seed=9)
    gm = gpu.Model.from_tensors(m)
    tr = oracle.Transducer(m)
    rng = np.random.default_rng(21)
    T_valid = [int(t) for t in rng.integers(0, 41, 21)]
    B, T_max = len(T_valid), 40
    enc = rng.standard_normal((B, T_max, cfg.d_model)).astype(np.float32)
    print(f"[decode] B={B} T={T_valid}", flush=True)
    d_enc = gpu.DeviceArray.from_numpy(enc, stream)
    got = gm.transducer_greedy(d_enc, T_valid, durations=durations, max_symbols=10, stream=stream)
    total = 0
    for b in range(B):
        ids, fr, cf, sp = tr.greedy(enc[b, :T_valid[b]], durations=durations, max_symbols=10)
        g_ids, g_fr, g_cf, g_sp = got[b]
        total += len(ids)
        assert np.array_equal(g_ids, ids), (b, g_ids[:20], ids[:20])
        assert np.array_equal(g_fr, fr) and np.array_equal(g_sp, sp)
        assert np.max(np.abs(g_cf - cf), initial=0.0) <= 1e-5
    print(f"[decode] {total} tokens identical over {B} items", flush=True)
    assert total > 20
    d_enc.free()


def test_greedy_decode_production_shape(gpu, stream):
    """The 0.6B decoder's shape: 2-layer LSTM of 640 (K = 1280 in the gate
    products, several register slabs per lane), joint 640, 1024 tokens + blank +
    5 durations (1030 outputs, not a multiple of 4), encoder width 1024, and 17
    ragged items (more than one LDS pass of 16)."""
    durations = (0, 1, 2, 3, 4)
    cfg = pm.Config(d_model=1024, n_layers=1, n_heads=8, ff_dim=256, n_mels=64, sub_channels=16, vocab_size=1024,
                    joint_hidden=640, pred_hidden=640, pred_rnn_layers=2, tdt_durations=durations)
    m = pm.add_prediction(pm.synthesize(cfg, "q8_0", heads=True, seed=640), seed=640)
    for n in ("joint.joint_net.2.weight", "joint.joint_net.2.bias"):
        t = m.tensors[n]
        m.tensors[n] = pm.Tensor(t.gtype, t.shape, (t.data * 60.0).astype(np.float32))
    gm = gpu.Model.from_tensors(m)
    tr = oracle.Transducer(m)
    rng = np.random.default_rng(17)
    T_valid = [125, 125, 3, 0, 64, 125, 99, 1, 125, 17, 80, 125, 42, 125, 7, 110, 125]
    B, T_max = len(T_valid), 125
    enc = rng.standard_normal((B, T_max, cfg.d_model)).astype(np.float32)
    print(f"[decode] production shape B={B} T={T_valid}", flush=True)
    d_enc = gpu.DeviceArray.from_numpy(enc, stream)
    got = gm.transducer_greedy(d_enc, T_valid, durations=durations, max_symbols=10, stream=stream)
    total = 0
    for b in range(B):
        ids, fr, cf, sp = tr.greedy(enc[b, :T_valid[b]], durations=durations, max_symbols=10)
        g_ids, g_fr, g_cf, g_sp = got[b]
        total += len(ids)
        assert np.array_equal(g_ids, ids), (b, g_ids[:20], ids[:20])
        assert np.array_equal(g_fr, fr) and np.array_equal(g_sp, sp)
        # The joint output is scaled x60 here, so logits reach a few hundred,
        # where one f32 ulp is 1.5e-5-3e-5; device and oracle sum the K = 640
        # products in different orders, so each logit may differ by a few ulps.
        # The confidence (N p - 1) / (N - 1), p = 1 / sum exp(l - l_max), moves
        # by at most ~2 max|dl| * p: 5e-5 covers two ulps at |l| ~ 256.
        assert np.max(np.abs(g_cf - cf), initial=0.0) <= 5e-5
    print(f"[decode] {total} tokens identical over {B} items", flush=True)
    assert total > 100
    d_enc.free()
    gm.close()


def _raw_greedy(gpu, gm, d_enc, T_valid, durations, blank, cap, stream):
    """pkx_transducer_greedy into arrays of -7: (ids, frames, conf, span) as [B][cap] and the counts."""
    B, T_max, _ = d_enc.shape
    ids, fr, sp = (np.full((B, cap), -7, np.int32) for _ in range(3))
    cf, cnt = np.full((B, cap), -7, np.float32), np.zeros(B, np.int32)
    tv, du = np.asarray(T_valid, np.int32), np.asarray(durations, np.int32)
    i32, f32 = C.POINTER(C.c_int32), C.POINTER(C.c_float)
    gpu.check(gpu.lib().pkx_transducer_greedy(
        gm.handle, d_enc.ptr, B, T_max, tv.ctypes.data_as(i32), du.ctypes.data_as(i32), len(du), blank, 10, cap,
        ids.ctypes.data_as(i32), fr.ctypes.data_as(i32), cf.ctypes.data_as(f32), sp.ctypes.data_as(i32),
        cnt.ctypes.data_as(i32), stream.handle))
    return (ids, fr, cf, sp), cnt


def test_greedy_decode_leaves_no_earlier_tokens(gpu, stream):
    """The outputs past an item's tokens are zeros, also after a call with more
    tokens whose records lay at the same place of the model's workspace."""
    durations = (0, 1, 2, 3, 4)
    cfg, m = _model(durations)
    gm = gpu.Model.from_tensors(m)
    enc = np.random.default_rng(5).standard_normal((3, 40, cfg.d_model)).astype(np.float32)
    d_enc = gpu.DeviceArray.from_numpy(enc, stream)
    most = None
    for T_valid in ([40, 40, 40], [3, 0, 11]):
        print(f"[decode] T={T_valid}", flush=True)
        out, cnt = _raw_greedy(gpu, gm, d_enc, T_valid, durations, cfg.vocab_size, 400, stream)
        for b in range(3):
            for a in out:
                assert not a[b, cnt[b]:].any(), (T_valid, b, cnt[b], a[b, cnt[b]:cnt[b] + 8])
        most = cnt if most is None else most
    assert (cnt < most).all()
    d_enc.free()


def _check_items(got, want, tol=1e-5):
    for b, (g, w) in enumerate(zip(got, want)):
        for i in (0, 1, 3):
            assert np.array_equal(g[i], w[i]), (b, i, g[i][:20], w[i][:20])
        assert np.max(np.abs(g[2] - w[2]), initial=0.0) <= tol


def test_greedy_decode_two_threads_one_model(gpu):
    """Two host threads decode different batches on one model, each on a stream
    of its own: the model's working memory goes to one call at a time, the
    other uses its own."""
    durations = (0, 1, 2, 3, 4)
    cfg, m = _model(durations, seed=3)
    gm, tr = gpu.Model.from_tensors(m), oracle.Transducer(m)
    rng = np.random.default_rng(33)
    jobs = []
    for B, T in ((3, 50), (18, 20)):
        enc = rng.standard_normal((B, T, cfg.d_model)).astype(np.float32)
        T_valid = [T] + [int(t) for t in rng.integers(0, T + 1, B - 1)]
        want = [tr.greedy(enc[b, :T_valid[b]], durations=durations, max_symbols=10) for b in range(B)]
        s = gpu.Stream()
        jobs.append((gpu.DeviceArray.from_numpy(enc, s), T_valid, want, s))
        s.sync()
    go, failed = threading.Barrier(2), []

    def work(job):
        d_enc, T_valid, want, s = job
        try:
            for call in range(8):
                go.wait(30)
                _check_items(gm.transducer_greedy(d_enc, T_valid, durations=durations, stream=s), want)
        except BaseException as e:   # noqa: BLE001 - reported by the test below
            failed.append(e)
            go.abort()

    print(f"[decode] two threads, T={[j[1] for j in jobs]}", flush=True)
    threads = [threading.Thread(target=work, args=(j,)) for j in jobs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed, failed
    for j in jobs:
        j[0].free()


def test_greedy_decode_past_the_kept_workspace(gpu, stream):
    """A call whose encoder projections alone exceed the 64 MB that stay with the
    model, then a small one."""
    durations = (0, 1, 2, 3, 4)
    cfg, m = _model(durations, seed=4)
    gm, tr = gpu.Model.from_tensors(m), oracle.Transducer(m)
    rng = np.random.default_rng(44)
    for B, T_max in ((16, 8300), (2, 30), (16, 8300)):
        T_valid = [int(t) for t in rng.integers(1, 31, B)]
        enc = np.zeros((B, T_max, cfg.d_model), np.float32)
        enc[:, :30] = rng.standard_normal((B, 30, cfg.d_model))
        print(f"[decode] B={B} T_max={T_max} T={T_valid}", flush=True)
        d_enc = gpu.DeviceArray.from_numpy(enc, stream)
        got = gm.transducer_greedy(d_enc, T_valid, durations=durations, cap=400, stream=stream)
        _check_items(got, [tr.greedy(enc[b, :T_valid[b]], durations=durations, max_symbols=10) for b in range(B)])
        d_enc.free()


def test_greedy_decode_more_items_than_a_grid_dimension(gpu, stream):
    """More 16-item blocks than a grid's second dimension holds (1,048,560 items):
    22 different items over and over, the repeats identical and the first ones
    the oracle's."""
    durations = (0, 1, 2, 3, 4)
    cfg, m = _model(durations, seed=6)
    gm, tr = gpu.Model.from_tensors(m), oracle.Transducer(m)
    n, B, cap = 22, 65535 * 16 + 40, 11
    one = np.random.default_rng(66).standard_normal((n, 1, cfg.d_model)).astype(np.float32)
    enc = np.concatenate([one] * (B // n) + [one[:B % n]])
    print(f"[decode] B={B}", flush=True)
    d_enc = gpu.DeviceArray.from_numpy(enc, stream)
    (ids, fr, cf, sp), cnt = _raw_greedy(gpu, gm, d_enc, [1] * B, durations, cfg.vocab_size, cap, stream)
    _check_items([(ids[b, :cnt[b]], fr[b, :cnt[b]], cf[b, :cnt[b]], sp[b, :cnt[b]]) for b in range(n)],
                 [tr.greedy(one[b], durations=durations, max_symbols=10) for b in range(n)])
    for a in (ids, fr, cf, sp, cnt[:, None]):
        rep = a[:B // n * n].reshape(B // n, n, -1)
        assert (rep == rep[:1]).all() and np.array_equal(a[B // n * n:], a[:B % n])
    d_enc.free()
