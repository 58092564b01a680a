"""The native host path (csrc/kvc_host.cpp) against the Python one: same
outputs and pool bytes for every form it accepts, None (the Python path) for
every other form, and the same exception types where a call is refused."""
import pytest
import torch

from nanovllm_amd import _native as nat
from nanovllm_amd.kernels.paged_attention import (decode_append_into, paged_decode_append,
                                                  paged_decode_attention)
from nanovllm_amd.layers.rotary import build_cos_sin_cache, qk_norm_rope_store

pytestmark = pytest.mark.gpu
DEV = "cuda"
PAGE, MAXB = 64, 4


class _Sub(torch.Tensor):
    pass


class _NeverNative:
    @staticmethod
    def decode(*_):
        return None

    @staticmethod
    def rope(*_):
        return None


def _calls(monkeypatch, fn, make):
    """fn on two equal sets of arguments, native then Python; (results,
    whether the native call served it)."""
    served = []
    real = nat.host()

    class Spy:
        @staticmethod
        def decode(*a):
            r = real.decode(*a)
            served.append(r is not None)
            return r

        @staticmethod
        def rope(*a):
            r = real.rope(*a)
            served.append(r is not None)
            return r

    out = []
    for host in (Spy, _NeverNative):
        monkeypatch.setattr(nat, "host", lambda h=host: h)
        args, kept = make()
        try:
            res = fn(*args)
        except Exception as e:  # noqa: BLE001
            res = type(e)
        out.append((res, kept))
    monkeypatch.undo()
    torch.cuda.synchronize()
    return out, any(served)


def _same(a, b):
    if isinstance(a, type) or isinstance(b, type):
        return a is b
    if a is None or b is None:
        return a is b
    if isinstance(a, (tuple, list)):
        return all(_same(x, y) for x, y in zip(a, b))
    return (a.shape == b.shape and a.stride() == b.stride() and a.dtype == b.dtype
            and torch.equal(a, b))


def _step(heads, kvh, batch, form):
    g = torch.Generator().manual_seed(heads * 100 + batch)
    dev = lambda t: t.to(DEV)  # noqa: E731
    bf = lambda *s: dev(torch.randn(*s, generator=g).to(torch.bfloat16))  # noqa: E731
    lens = torch.randint(1, MAXB * PAGE + 1, (batch,), generator=g)
    tables = torch.randperm(batch * MAXB, generator=g).view(batch, MAXB)
    slots = tables[torch.arange(batch), (lens - 1) // PAGE] * PAGE + (lens - 1) % PAGE
    kc, vc = bf(batch * MAXB, PAGE, kvh, 128), bf(batch * MAXB, PAGE, kvh, 128)
    qkv = bf(batch, (heads + 2 * kvh) * 128)
    q, k, v = qkv.split((heads * 128, kvh * 128, kvh * 128), dim=-1)
    q, k, v = q.unflatten(-1, (heads, 128)), k.unflatten(-1, (kvh, 128)), v.unflatten(-1, (kvh, 128))
    a = {"q": q, "k": k, "v": v, "kc": kc, "vc": vc, "slots": dev(slots.int()),
         "bt": dev(tables.int()), "lens": dev(lens.int()), "scale": 128 ** -0.5}
    if form == "dense":
        a.update(q=q.contiguous(), k=k.contiguous(), v=v.contiguous())
    elif form == "slots64":
        a["slots"] = a["slots"].long()
    elif form == "heads-first q":         # [heads, batch, 128] storage
        a["q"] = q.transpose(0, 1).contiguous().transpose(0, 1)
    elif form == "wide tables":           # a row stride past its width
        a["bt"] = dev(torch.cat([tables, tables], 1).int())[:, :MAXB]
    elif form == "lens64":
        a["lens"] = a["lens"].long()
    elif form == "tables64":
        a["bt"] = a["bt"].long()
    elif form == "strided slots":
        a["slots"] = a["slots"].repeat_interleave(2)[::2]
    elif form == "transposed tables":
        a["bt"] = a["bt"].t().contiguous().t()
    elif form == "int scale":
        a["scale"] = 1
    elif form == "dims apart":            # q with a dim stride of 2
        a["q"] = q.repeat_interleave(2, -1)[..., ::2]
    elif form == "subclass":
        a["q"] = q.as_subclass(_Sub)
    elif form == "odd q rows":            # 4-byte aligned: refused
        a["q"] = torch.nn.functional.pad(q.reshape(batch, -1), (2, 0))[:, 2:].unflatten(-1, (heads, 128))
    elif form == "fp16 q":
        a["q"] = q.half()
    elif form == "split pool":            # a pool that is not contiguous
        a["kc"] = torch.cat([kc, kc], 2)[:, :, :kvh]
    elif form == "short v pool":
        a["vc"] = vc[:-1]
    else:
        assert form == "views"
    return a


NATIVE = ["views", "dense", "slots64", "heads-first q", "wide tables"]
PYTHON = ["lens64", "tables64", "strided slots", "transposed tables", "int scale", "dims apart",
          "subclass"]
REFUSED = ["odd q rows", "fp16 q", "split pool", "short v pool"]


@pytest.mark.parametrize("form", NATIVE + PYTHON + REFUSED)
@pytest.mark.parametrize("heads,kvh,batch", [(32, 4, 5), (16, 2, 1), (16, 8, 3), (6, 1, 2)])
@pytest.mark.parametrize("append", [True, False])
def test_decode_forms(monkeypatch, heads, kvh, batch, form, append):
    print(f"[host] decode {heads}/{kvh} batch {batch} {form} append={append}", flush=True)

    def make():
        a = _step(heads, kvh, batch, form)
        kept = [a["kc"], a["vc"]]
        if append:
            return (a["q"], a["k"], a["v"], a["kc"], a["vc"], a["slots"], a["bt"], a["lens"],
                    a["scale"]), kept
        return (a["q"], a["kc"], a["vc"], a["bt"], a["lens"], a["scale"], MAXB * PAGE), kept

    fn = paged_decode_append if append else paged_decode_attention
    (native, python), served = _calls(monkeypatch, fn, make)
    if form in NATIVE or (form == "strided slots" and (batch == 1 or not append)) \
            or (form == "transposed tables" and batch == 1):
        assert served
    elif form not in REFUSED:
        assert not served
    assert isinstance(native[0], type) == (form in REFUSED)
    assert _same(native[0], python[0])
    assert _same(native[1], python[1])


@pytest.mark.parametrize("form", ["views", "positions32", "no weights", "no cache", "weights32",
                                  "strided positions", "no value", "half table"])
@pytest.mark.parametrize("tokens", [1, 37])
@pytest.mark.parametrize("return_k", [True, False])
def test_rope_forms(monkeypatch, tokens, form, return_k):
    heads, kvh = 16, 8
    print(f"[host] rope tokens {tokens} {form} return_k={return_k}", flush=True)

    def make():
        g = torch.Generator().manual_seed(tokens)
        bf = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16).to(DEV)  # noqa: E731
        qkv = bf(tokens, (heads + 2 * kvh) * 128)
        q, k, v = qkv.split((heads * 128, kvh * 128, kvh * 128), dim=-1)
        q, k, v = q.unflatten(-1, (heads, 128)), k.unflatten(-1, (kvh, 128)), v.unflatten(-1, (kvh, 128))
        pos = torch.randint(0, 512, (tokens,), generator=g).to(DEV)
        cs = build_cos_sin_cache(128, 512, 1e6, DEV)
        w = [bf(128), bf(128)]
        kc, vc = bf(4, PAGE, kvh, 128), bf(4, PAGE, kvh, 128)
        slots = torch.randperm(4 * PAGE, generator=g)[:tokens].to(torch.int32).to(DEV)
        if form == "positions32":
            pos = pos.int()
        elif form == "strided positions":
            pos = pos.repeat_interleave(2)[::2]
        elif form == "no weights":
            w = [None, None]
        elif form == "weights32":
            w = [x.float() for x in w]
        elif form == "half table":
            cs = cs.half()
        kept = [kc, vc]
        if form in ("no cache", "no value"):
            return (q, k, None if form == "no value" else v, pos, cs, *w, 1e-6, None, None, None,
                    return_k), kept
        return (q, k, v, pos, cs, *w, 1e-6, kc, vc, slots, return_k), kept

    (native, python), served = _calls(monkeypatch, qk_norm_rope_store, make)
    if form in ("weights32", "half table") or (form == "strided positions" and tokens > 1):
        assert not served
    else:
        assert served
    assert isinstance(native[0], type) == (form == "half table")
    assert _same(native[0], python[0])
    assert _same(native[1], python[1])


def test_rope_refuses_a_v_pool_alone():
    q, k, v = (torch.zeros(3, h, 128, dtype=torch.bfloat16, device=DEV) for h in (16, 8, 8))
    pos = torch.arange(3, device=DEV)
    cs = build_cos_sin_cache(128, 16, 1e6, DEV)
    pool = torch.zeros(1, PAGE, 8, 128, dtype=torch.bfloat16, device=DEV)
    print("[host] rope with a v pool alone", flush=True)
    with pytest.raises(ValueError, match="both caches"):
        qk_norm_rope_store(q, k, v, pos, cs, v_cache=pool, slot_mapping=pos.int())
    with pytest.raises(ValueError, match="v_cache"):
        qk_norm_rope_store(q, k, v, pos, cs, k_cache=pool, slot_mapping=pos.int())


@pytest.mark.parametrize("heads,kvh,batch", [(32, 4, 5), (16, 2, 1), (16, 8, 3), (6, 1, 2)])
@pytest.mark.parametrize("view", [False, True])
def test_decode_into_a_given_output(monkeypatch, heads, kvh, batch, view):
    print(f"[host] decode into output {heads}/{kvh} batch {batch} view={view}", flush=True)

    def make():
        a = _step(heads, kvh, batch, "views")
        out = torch.full((batch + 1, heads + 2, 128), 7.0, dtype=torch.bfloat16, device=DEV)
        given = out[:batch, 1:heads + 1] if view else out[:batch, :heads].contiguous()
        return (given, a["q"], a["k"], a["v"], a["kc"], a["vc"], a["slots"], a["bt"], a["lens"],
                a["scale"]), [out, a["kc"], a["vc"]]

    (native, python), served = _calls(monkeypatch, decode_append_into, make)
    assert served
    assert _same(native[0], python[0]) and _same(native[1], python[1])
    args, kept = make()
    assert decode_append_into(*args) is args[0]
    want = paged_decode_append(*make()[0][1:])
    assert torch.equal(args[0], want)
    if view:                                   # nothing around the view is written
        kept[0][:batch, 1:heads + 1] = 7.0
        assert bool((kept[0] == 7.0).all())


@pytest.mark.parametrize("call", ["rope", "decode", "append"])
def test_out_of_memory_is_torchs_error(call):
    # An allocation that fails before a launch leaves the call to the Python
    # function, which raises torch's own error; the next call works.
    # One row repeated: an output of 550 GB, which no card holds.
    n = 1 << 26
    q, k, v = (torch.zeros(1, h, 128, dtype=torch.bfloat16, device=DEV).expand(n, h, 128)
               for h in (32, 4, 4))
    pool = torch.zeros(1, PAGE, 4, 128, dtype=torch.bfloat16, device=DEV)
    ints = torch.ones(n, dtype=torch.int32, device=DEV)
    cs = build_cos_sin_cache(128, 16, 1e6, DEV)

    def run(m):
        t = ints[:m]
        if call == "rope":
            return qk_norm_rope_store(q[:m], k[:m], v[:m], t, cs)
        if call == "decode":
            return paged_decode_attention(q[:m], pool, pool, t.view(m, 1) - 1, t, 0.1, 1)
        return paged_decode_append(q[:m], k[:m], v[:m], pool, pool, t - 1, t.view(m, 1) - 1, t, 0.1)

    run(2)
    print(f"[host] out of memory: {call}", flush=True)
    with pytest.raises(torch.OutOfMemoryError):
        run(n)
    run(2)
    torch.cuda.synchronize()
