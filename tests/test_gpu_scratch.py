"""GPU tests of the device's shared scratch (scratch.py): calls on two streams with no
synchronisation of their own are ordered through the buffer and give the single-stream bits,
a grown buffer stays valid for work queued on every stream that used it, split-K partials
handed out in the scratch are refused once it has been reused, and threads take it in turn."""

import threading

import pytest
import torch

from oracle import q8

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _pair(pkg, L, seed):
    z, _, po, pi = pkg.workloads.pair_inputs(L, 128, 128, seed=seed, dtype=torch.float16)
    T = pkg.trimul
    return z.to(DEV), T.TriMulPair(T.TriMul.from_weights(po, device=DEV), T.TriMul.from_weights(pi, device=DEV))


def test_two_streams_are_ordered_through_the_scratch(gpu_lib, pkg):
    cases = [_pair(pkg, L, seed) for L, seed in ((96, 1), (160, 2), (64, 3))]
    refs = [m(z) for z, m in cases]
    torch.cuda.synchronize()
    pkg.scratch.release(DEV)  # start small: the calls below grow the buffer while streams alternate
    s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()
    outs = []
    for rep in range(3):
        for k, (z, m) in enumerate(cases):
            with torch.cuda.stream(s1 if (rep + k) % 2 == 0 else s2):
                outs.append((k, m(z)))
    torch.cuda.synchronize()
    for k, out in outs:
        assert torch.equal(out.view(torch.int16), refs[k].view(torch.int16)), k


def test_stale_partials_are_refused(gpu_lib, pkg):
    x, qq, s, b = q8.make_q8_inputs(238, 10240, 2560, seed=4)
    lin = pkg.q8.Q8Linear(torch.from_numpy(qq), torch.from_numpy(s), torch.from_numpy(b))
    xt = torch.from_numpy(x).to(DEV)
    D = 2560
    res = torch.randn(238, D, device=DEV)
    w, bb = torch.ones(D, device=DEV), torch.zeros(D, device=DEV)
    parts = lin.partials(xt)
    assert parts[1] > 1  # split-K at this shape: the partials live in the scratch
    pkg.kernels.esmc_layer_norm(res, w, bb, 1e-5, y_parts=parts)  # consumed in time: fine
    lin(xt)  # another scratch user
    with pytest.raises(RuntimeError, match="stale"):
        pkg.kernels.esmc_layer_norm(res, w, bb, 1e-5, y_parts=parts)


def _users(pkg):
    """(name, native entry point, call) of everything that takes the scratch, at shapes that do."""
    K, T = pkg.kernels, pkg.trimul
    z, pair = _pair(pkg, 40, 5)
    x, qq, s, b = (torch.from_numpy(a) for a in q8.make_q8_inputs(40, 2048, 2560, seed=6))
    lin, x = pkg.q8.Q8Linear(qq, s, b), x.to(DEV)
    gated = pkg.q8.Q8Linear(qq, s, b).swiglu_pairs()
    g = torch.Generator().manual_seed(7)
    w = lambda *shape: torch.randn(*shape, generator=g).to(DEV) * 0.05  # noqa: E731
    zw = torch.randn(1, 30, 30, 256, generator=g).to(DEV).half()
    tr = pkg.trunk.PairTransition(w(256), w(256), w(1024, 256), w(256, 1024), w2=w(1024, 256))
    q = [q8.make_q8_inputs(1, k, n, seed=n)[1:] for k, n in ((256, 768), (256, 256), (256, 640), (320, 256))]
    lins = [pkg.q8.Q8Linear(*(torch.from_numpy(a) for a in t)) for t in q]
    blk = pkg.esmc.EsmcBlock(*(w(256) for _ in range(6)), *lins, 4)
    xb, xr = torch.randn(1, 9, 256, generator=g).to(DEV), torch.randn(40, 2560, generator=g).to(DEV)
    ones, zeros = torch.ones(2560, device=DEV), torch.zeros(2560, device=DEV)
    assert K.q8_workspace_bytes(40, 2048, 2560) > 0
    return [
        ("update", "tmu_forward_ws", lambda: pair.t_out(z)),
        ("pair", "tmu_pair_forward_ws", lambda: pair(z)),
        ("transition", "pair_transition_ws", lambda: tr(zw)),
        ("linear", "q8_linear_packed_ws", lambda: lin(x)),
        ("linear, 3-d", "q8_linear_packed_ws", lambda: lin(x[None])),
        ("gated linear", "q8_linear_swiglu_packed_ws", lambda: gated.swiglu(x)),
        ("partials", "q8_linear_packed_partials", lambda: lin.partials(x)[0].clone()),
        ("partials' consumer", "esmc_layer_norm_parts",
         lambda: K.esmc_layer_norm(xr.clone(), ones, zeros, 1e-5, y_parts=lin.partials(x))),
        ("language model block", "esmc_block", lambda: blk(xb)),
    ]


@pytest.mark.parametrize("which", range(9))
def test_the_scratch_is_held_until_the_launches_are_queued(gpu_lib, pkg, monkeypatch, which):
    # another thread that asks for the scratch while a native call is about to queue its launches gets it only
    # behind that call: its own launches would otherwise land between them
    name, entry, call = _users(pkg)[which]
    ref = call()
    real, seen = pkg.capi.lib(), []

    class Lib:
        def __getattr__(self, n):
            f = getattr(real, n)
            if n != entry:
                return f

            def native(*args):
                done = threading.Event()

                def other():
                    with pkg.scratch.guard(DEV):
                        pkg.scratch.get(1 << 16, DEV)
                    done.set()

                t = threading.Thread(target=other)
                t.start()
                early = done.wait(0.3)
                rc = f(*args)
                seen.append((early, done, t))
                return rc

            return native

    monkeypatch.setattr(pkg.capi, "lib", lambda *a, **k: Lib())
    out = call()
    monkeypatch.undo()
    assert len(seen) == 1, name
    early, done, t = seen[0]
    t.join(5)
    assert done.is_set() and not early, name
    assert torch.equal(out, ref), name


def test_threads_on_one_stream_and_on_their_own(gpu_lib, pkg):
    # two threads that run different scratch users again and again: every result has the bits of one thread alone
    users = [u for u in _users(pkg) if u[0] in ("language model block", "pair", "linear", "transition")]
    refs = [call() for _, _, call in users]
    torch.cuda.synchronize()
    for own in (False, True):
        wrong = []

        def work(k):
            stream = torch.cuda.Stream() if own else torch.cuda.default_stream()
            with torch.cuda.stream(stream):
                outs = [(i, users[i][2]()) for n in range(20) for i in [(k + n) % len(users)]]
                stream.synchronize()
            wrong.extend(users[i][0] for i, o in outs if not torch.equal(o, refs[i]))

        threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not wrong, (own, wrong)
