"""K-quant batches under HIP graph capture that the matrix cores take and the thin kernels hold: their scratch buffer grows where
it would have done for the thin kernels, with the bits of the same call outside of a capture; elsewhere it does not grow.  And an allocation that fails."""
import ctypes as C

import numpy as np
import pytest

import oracle as fo
from test_gpu_parity import bits, fa, make_weights, to_dev  # noqa: F401 (fa: the module's fixture)

pytestmark = pytest.mark.gpu


def _new_stream(fa):
    """A stream that no call has run on (torch hands out the streams of a pool again)."""
    import torch
    handle = C.c_void_p()
    assert fa.lib().hipStreamCreateWithFlags(C.byref(handle), 1) == 0
    return torch.cuda.ExternalStream(handle.value)


def _captured(fa, call, out, eager, between):
    """`call` captured on a stream that has run `between` only; every replay against `eager`, bit for bit."""
    import torch
    stream = _new_stream(fa)
    with torch.cuda.stream(stream):
        if between is not None:
            between()
        stream.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=stream):
            call()
        for rep in range(3):
            for o in out:
                o.zero_()
            g.replay()
            stream.synchronize()
            for o, e in zip(out, eager):
                assert np.array_equal(bits(o.cpu().numpy()), bits(e.cpu().numpy())), rep
            if between is not None:  # (the stream's own calls, and another's, between the replays)
                between()
            with torch.cuda.stream(torch.cuda.Stream()):
                call()
            torch.cuda.synchronize()


def test_quantized_batches_on_a_stream_without_scratch_memory(fa):
    """17 rows of a Q4_K 4096 x 4096 matrix: in frk_hip_gemm_q8k_dev and frk_hip_gemm_acts_dev the thin kernels need no scratch
    memory, so both are captured on a stream that has none; frk_hip_gemm_dev, whose quantization always needs some, is not."""
    import torch
    from frink_amd import synth
    rows = cols = 4096
    w = fa.Weights.from_host(fo.Q4_K, make_weights(fo.Q4_K, rows, cols, seed=71), rows, cols)
    x = to_dev(synth.activations(72, 17, cols))
    eager = w.gemm(x)
    q, d, bs = fa.quantize_q8_k(x.reshape(-1))
    acts = fa.BatchActs(17, cols)
    acts.quantize(x)
    y = torch.zeros_like(eager)
    torch.cuda.synchronize()
    print("q8k", flush=True)
    _captured(fa, lambda: w.gemm_q8k((q, d, bs), 17, out=y), [y], [eager], None)
    print("acts", flush=True)
    _captured(fa, lambda: w.gemm_acts(acts, out=y), [y], [eager], None)
    y, beyond, xb = torch.zeros_like(eager), torch.zeros((65, rows), device="cuda"), to_dev(synth.activations(75, 65, cols))
    acts65 = fa.BatchActs(65, cols)
    acts65.quantize(xb)
    # (the last one is split, and beyond what the thin kernels hold)
    for what, call, out in (("gemm", lambda: w.gemm(x, out=y), y), ("beyond", lambda: w.gemm(xb, out=beyond), beyond),
                            ("acts beyond", lambda: w.gemm_acts(acts65, out=beyond), beyond)):
        print(what, flush=True)
        torch.cuda.synchronize()
        with pytest.raises(fa.BackendError) as e:
            with torch.cuda.graph(torch.cuda.CUDAGraph(), stream=_new_stream(fa)):
                call()
        assert e.value.code == fa.ERR_HIP
        torch.cuda.synchronize()
        assert not out.any()
    w.release()


def test_batches_on_a_stream_whose_scratch_buffer_is_too_small(fa):
    """40 rows of a Q6_K 4096 x 7168 matrix: 5.5 MiB of scratch memory, on a stream whose buffer has the smallest size (4 MiB) from a
    call of two rows."""
    import torch
    from frink_amd import synth
    rows, cols = 4096, 7168
    data = make_weights(fo.Q6_K, 64, cols, seed=73)
    data = np.concatenate([np.roll(data.reshape(64, -1), i, axis=0).reshape(-1) for i in range(rows // 64)])
    w = fa.Weights.from_host(fo.Q6_K, data, rows, cols)
    x = to_dev(synth.activations(74, 40, cols))
    eager = w.gemm(x)
    pair = [e.clone() for e in fa.gemm_pair(w, w, x)]
    y, y2 = torch.zeros_like(eager), [torch.zeros_like(e) for e in pair]
    torch.cuda.synchronize()
    print("gemm", flush=True)
    _captured(fa, lambda: w.gemm(x, out=y), [y], [eager], lambda: w.gemm(x[:2]))
    print("pair", flush=True)
    _captured(fa, lambda: fa.gemm_pair(w, w, x, outs=y2), y2, pair, lambda: w.gemm(x[:2]))
    w.release()


def test_a_failed_allocation_is_reported_once(fa):
    """More memory than any device has: an error, and the next calls on the thread are not told of it again."""
    import torch
    from frink_amd import synth
    w = fa.Weights.from_host(fo.Q4_K, make_weights(fo.Q4_K, 64, 512, seed=76), 64, 512)
    x = to_dev(synth.activations(77, 3, 512))
    want = w.gemm(x).clone()
    torch.cuda.synchronize()
    with pytest.raises(fa.BackendError) as e:
        fa.BatchActs(10 ** 10, 32768)
    assert e.value.code in (fa.ERR_HIP, fa.ERR_OOM)
    got = w.gemm(x)
    torch.cuda.synchronize()
    assert np.array_equal(bits(got.cpu().numpy()), bits(want.cpu().numpy()))
    w.release()
