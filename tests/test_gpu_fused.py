"""GPU parity: the fused entry points on unpacked codes (hkv_fused_decode,
hkv_fused_forward behind fused_dequant_attn_decode / _forward) against the float64 oracle."""
import math

import numpy as np
import pytest
import torch

from oracle import attention as oa
from oracle import compressor as oc

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
TOL = 2e-3   # the decode and prefill tests' bound


def _inputs(seed, B, Hq, Hkv, S, Sq, dtype):
    g = torch.Generator().manual_seed(seed)
    K = torch.randn((B, Hkv, S, 128), generator=g)
    K[..., [7, 31, 64, 100]] *= 8
    V = torch.randn((B, Hkv, S, 128), generator=g)
    q = (torch.randn((B, Hq, Sq, 128), generator=g) / math.sqrt(128)).to(dtype)
    kc, ks, kz = oc.compress(K.half().numpy(), 128)
    vc, vs, vz = oc.compress(V.half().numpy(), 128)
    shape = (B, Hkv, S)
    return q, kc, ks.reshape(shape), kz.reshape(shape), vc, vs.reshape(shape), vz.reshape(shape)


def _reference(q, kc, ks, kz, vc, vs, vz):
    return np.stack([oa.attend(q[b].double().numpy(), oa.dequant_rows(kc[b], ks[b], kz[b]),
                               oa.dequant_rows(vc[b], vs[b], vz[b])) for b in range(q.shape[0])])


def _check(out, ref, dtype):
    got = out.float().cpu().numpy()
    assert np.all(np.isfinite(got))
    # plus the output's own rounding, half a unit in the last place: 2^-8 of the value for the
    # 8 significant bits of bf16, 2^-11 for fp16 (few keys: outputs of several units)
    tol = TOL + np.abs(ref) * 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    err = np.abs(got - ref)
    print("  max abs err %.3e" % err.max(), flush=True)
    assert np.all(err <= tol)


def _dev(x):
    return torch.from_numpy(np.ascontiguousarray(x)).to(DEV)


# rows of a block, of a tile and of a range that end everywhere, multiples of 4 and not
@pytest.mark.parametrize("S", [1, 3, 15, 16, 17, 64, 65, 127, 1000, 2049])
@pytest.mark.parametrize("B,hq,hkv", [(1, 4, 4), (2, 14, 2), (1, 16, 1)])
def test_fused_edges(B, hq, hkv, S):
    from heterokv import fused_dequant_attn_decode, fused_dequant_attn_forward
    for Sq, dtype in ((1, torch.float16), (1, torch.bfloat16), (37, torch.float16), (130, torch.bfloat16)):
        print("case: fused B=%d %d/%d S=%d Sq=%d %s" % (B, hq, hkv, S, Sq, dtype), flush=True)
        x = _inputs(1000 + S, B, hq, hkv, S, Sq, dtype)
        args = (x[0].to(DEV),) + tuple(_dev(t) for t in x[1:])
        fn = fused_dequant_attn_decode if Sq == 1 else fused_dequant_attn_forward
        _check(fn(*args), _reference(*x), dtype)


@pytest.mark.parametrize("Sq", [1, 20])
def test_fused_input_forms(Sq):
    """Float zero points, codes with their high bits set, strided and unaligned views, a
    two-dimensional single head, float32 queries and no token at all."""
    from heterokv import fused_dequant_attn_decode, fused_dequant_attn_forward
    fn = fused_dequant_attn_decode if Sq == 1 else fused_dequant_attn_forward
    print("case: fused input forms Sq=%d" % Sq, flush=True)
    x = _inputs(5, 1, 2, 2, 90, Sq, torch.float16)
    q, kc, ks, kz, vc, vs, vz = x
    ref = _reference(*x)
    a = [q.to(DEV)] + [_dev(t) for t in x[1:]]
    _check(fn(a[0], a[1], a[2], a[3].float(), a[4], a[5], a[6].float()), ref, torch.float16)
    _check(fn(a[0], a[1] | 0xA0, *a[2:4], a[4] | 0x50, *a[5:]), ref, torch.float16)
    _check(fn(a[0].float(), *a[1:]), ref, torch.float16)
    odd = [torch.cat([t.new_zeros(1), t.reshape(-1)])[1:].view(t.shape) for t in a[1:]]   # bases off by one element
    _check(fn(a[0], *odd), ref, torch.float16)
    wide = [torch.stack([t, t], -1)[..., 0] for t in a[1:]]                               # strided views
    _check(fn(a[0], *wide), ref, torch.float16)
    one = fn(a[0][:, :1], a[1][0, 0], a[2][0, 0], a[3][0, 0], a[4][0, 0], a[5][0, 0], a[6][0, 0])
    _check(one, ref[:, :1], torch.float16)
    none = fn(a[0], *[t[:, :, :0] for t in a[1:]])
    assert none.shape == a[0].shape and not none.any()


@pytest.mark.parametrize("hkv,S,Sq", [(4, 9000, 20), (1, 5003, 200)])
def test_fused_forward_split_keys(hkv, S, Sq):
    """Few queries over many keys: split over workgroups and combined."""
    from heterokv import fused_dequant_attn_forward
    print("case: fused forward split %d heads S=%d Sq=%d" % (hkv, S, Sq), flush=True)
    x = _inputs(9, 1, hkv, hkv, S, Sq, torch.float16)
    _check(fused_dequant_attn_forward(x[0].to(DEV), *[_dev(t) for t in x[1:]]), _reference(*x), torch.float16)


@pytest.mark.parametrize("hq,hkv,S,Sq", [(12, 1, 70, 255), (12, 1, 70, 256), (12, 1, 33, 257)])
def test_fused_forward_row_rule(hq, hkv, S, Sq, monkeypatch):
    """Query rows per kv head around 3072, those from there on with the codes repacked (into a
    pool whose last block is written only in part), as calls with many more keys have it."""
    from heterokv import fused_dequant_attn_forward, ops
    monkeypatch.setattr(ops, "_repacks", lambda b, qh, kh, queries, tokens: queries * qh >= 3072 * kh)
    assert ops._repacks(2, hq, hkv, Sq, S) == (Sq >= 256)
    print("case: fused forward rows %d" % (hq // hkv * Sq), flush=True)
    x = _inputs(11, 2, hq, hkv, S, Sq, torch.float16)
    _check(fused_dequant_attn_forward(x[0].to(DEV), *[_dev(t) for t in x[1:]]), _reference(*x), torch.float16)


def test_fused_decode_on_two_streams():
    """Overlapping calls on two streams, neither ordered after the other: every result against
    the oracle (with one workspace they would mix their partial states)."""
    from heterokv import fused_dequant_attn as fda
    print("case: fused decode on two streams", flush=True)
    xs = [_inputs(21 + i, 1, 8, 8, 3000 + 500 * i, 1, torch.float16) for i in range(2)]
    args = [(x[0].to(DEV),) + tuple(_dev(t) for t in x[1:]) for x in xs]
    refs = [_reference(*x) for x in xs]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(DEV) for _ in range(2)]
    outs = [[], []]
    for _ in range(20):
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                outs[i].append(fda.fused_dequant_attn_decode(*args[i]))
    torch.cuda.synchronize()
    keys = {(torch.device(DEV), s.cuda_stream) for s in streams}
    assert keys <= set(fda._WS) and len({id(fda._WS[k]) for k in keys}) == 2
    for i in range(2):
        for o in outs[i]:
            _check(o, refs[i], torch.float16)
    fda.check_errors(DEV)


def test_fused_decode_captured_call():
    """A captured call's replays, with new queries and with eager calls on other streams between
    them (the graph clears and owns its workspace), against the oracle."""
    from heterokv import fused_dequant_attn as fda
    print("case: fused decode in a graph", flush=True)
    x = _inputs(31, 1, 8, 8, 2500, 1, torch.float16)
    q = x[0].to(DEV)
    args = tuple(_dev(t) for t in x[1:])
    fda.fused_dequant_attn_decode(q, *args)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = fda.fused_dequant_attn_decode(q, *args)
    side = torch.cuda.Stream(DEV)
    for scale in (1.0, -0.5, 2.0, 0.25):
        q.copy_(x[0] * scale)
        ref = _reference(x[0] * scale, *x[1:])
        torch.cuda.synchronize()
        graph.replay()
        with torch.cuda.stream(side):
            eager = fda.fused_dequant_attn_decode(q, *args)
        torch.cuda.synchronize()
        _check(out, ref, torch.float16)
        _check(eager, ref, torch.float16)
