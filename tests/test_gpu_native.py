"""The native call path (flydsl_amd/csrc/launch.cpp) against the Python
launchers it stands for: the same bits for every form of call both take, and
None (so that the Python launcher does the call, or raises) for the rest."""

from __future__ import annotations

import pytest
import torch

import flydsl_amd.pa_decode as pd
from flydsl_amd import (_lib, build_fused_rope_cache_module, flydsl_mla_fwd_decode, flydsl_qk_norm_rope_quant,
                        get_mla_metadata_info_v1, get_mla_metadata_v1, get_pa_metadata, mla_reduce_v1,
                        pa_decode_ps_launch, workloads)
from tests._cases import make_case
from tests.test_gpu_parity import to_dev

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def both(monkeypatch, call):
    """call() by the native path -- which must take it -- and by Python."""
    native = _lib.native()
    assert native is not None
    taken = []

    class Spy:
        def __getattr__(self, name):
            def f(*args):
                r = getattr(native, name)(*args)
                taken.append(r is not None)
                return r
            return f

    monkeypatch.setattr(_lib, "_NATIVE", Spy())
    got = call()
    torch.cuda.synchronize()
    assert taken and all(taken)
    monkeypatch.setattr(_lib, "_NATIVE", False)
    want = call()
    torch.cuda.synchronize()
    monkeypatch.setattr(_lib, "_NATIVE", native)
    for g, w in zip(got, want):
        assert (g is None and w is None) or (isinstance(g, str) and g == w) or torch.equal(
            g.view(torch.uint8) if g.element_size() == 1 else g, w.view(torch.uint8) if w.element_size() == 1 else w)


def strided(t, dims):
    """A copy of t whose dims have room between their entries."""
    shape = [2 * n if i in dims else n for i, n in enumerate(t.shape)]
    big = torch.zeros(shape, dtype=t.dtype, device=t.device)
    view = big[tuple(slice(0, n) for n in t.shape)]
    view.copy_(t)
    return view


DECODE = {
    "owner": dict(batch=3, ctx=[1, 40, 500]),
    "split_gqa8_pt": dict(batch=2, num_query_heads=16, ctx=[3000, 9], per_token=True),
    "team_gqa8": dict(batch=150, num_query_heads=64, num_kv_heads=8, ctx=[20000] + [30] * 149),
    "balanced_gqa4_pt": dict(batch=150, num_query_heads=32, num_kv_heads=8, ctx=[20000] + [30] * 149, per_token=True),
    "coop": dict(batch=3, query_length=4, num_query_heads=64, num_kv_heads=4, block_size=64, ctx=[4, 900, 5000]),
    "d64_slots": dict(batch=3, head_size=64, ctx=[1, 700, 4000]),
    "window": dict(batch=3, ctx=[5, 400, 3000], sliding_window=500),
    "p1024": dict(batch=3, block_size=1024, ctx=[5, 3000, 700]),
}


@pytest.mark.parametrize("form", ["plain", "strided", "f16_partials", "plain_v_p0"])
@pytest.mark.parametrize("name", sorted(DECODE))
def test_decode_native_equals_python(name, form, monkeypatch):
    case = to_dev(make_case(seed=len(name), **DECODE[name]))
    q, kc, vc, ks, vs = (case[k] for k in ("query", "key_cache", "value_cache", "key_scale", "value_scale"))
    hkv, bs = kc.shape[1], kc.shape[3]
    gqa, ql, d, b = q.shape[1] // hkv, case["query_length"], q.shape[2], case["context_lengths"].shape[0]
    kw = {}
    out_dtype = torch.bfloat16
    if form == "strided":
        q, kc, vc = strided(q, (0, 1)), strided(kc.view(torch.uint8), (0, 1)).view(kc.dtype), strided(
            vc.view(torch.uint8), (0,)).view(vc.dtype)
        if ks.dim() > 1:
            ks, vs = strided(ks, (0, 1)), strided(vs, (0, 1))
        out_dtype = torch.float32
    elif form == "f16_partials":
        q = q.half()
        P = max(4, pd.get_recommended_splits(b, hkv, sliding_window=case["sliding_window"], query_length=ql)
                if case["sliding_window"] else 4)
        if bs != 1024:
            es = torch.zeros(b, hkv, P, ql * gqa, device=DEV)
            kw = dict(exp_sums=es, max_logits=es.clone(), max_context_partition_num=P,
                      temporary_output=torch.zeros(b, hkv, P, ql * gqa, d, device=DEV))
    elif form == "plain_v_p0" and d == 128:
        nb = vc.shape[0]
        vc = vc.view(torch.uint8).permute(0, 1, 3, 2, 4).reshape(nb, hkv, d, bs).contiguous().view(vc.dtype)
    bt, pages, indptr = case["block_tables"], None, None
    if bs == 1024:
        ctx = case["context_lengths"].tolist()
        rows = [bt[i, : -(-c // bs)] for i, c in enumerate(ctx)]
        pages = torch.cat(rows)
        indptr = torch.tensor([0] + [len(r) for r in rows]).cumsum(0).to(torch.int32).to(DEV)
        kw["metadata"] = get_pa_metadata(q, kc, case["context_lengths"], indptr, q.shape[1], hkv)
        bt = None

    def call():
        out = torch.zeros(q.shape, dtype=out_dtype, device=DEV)
        if form == "strided":
            out = strided(out, (1,))
        route = pa_decode_ps_launch(out, q, kc, vc, case["context_lengths"], pages, indptr, case["softmax_scale"], ks,
                                    vs, sliding_window=case["sliding_window"], block_tables=bt, **kw)
        return route, out.clone()

    both(monkeypatch, call)


@pytest.mark.parametrize("layout", ["flash", "atom", "trans"])
@pytest.mark.parametrize("dtype,fp8,i64,reuse", [("bf16", True, False, True), ("f16", False, True, False)])
def test_rope_native_equals_python(layout, dtype, fp8, i64, reuse, monkeypatch):
    T, qh, kh, d, bs, nb = 37, 6, 2, 64, 16, 8
    g = torch.Generator(device=DEV).manual_seed(3)
    dt = torch.bfloat16 if dtype == "bf16" else torch.float16
    rand = lambda *s: torch.randn(*s, generator=g, device=DEV).to(dt)
    q, k, v = strided(rand(T, qh, d), (0,)), rand(T, kh, d), rand(T, kh, d)
    cos, sin = rand(50, d // 2 if reuse else d), rand(50, d // 2 if reuse else d)
    it = torch.int64 if i64 else torch.int32
    pos = torch.randint(0, 50, (T,), generator=g, device=DEV).to(it)
    slots = torch.randperm(nb * bs, generator=g, device=DEV)[:T].to(it)
    cdt = torch.uint8 if fp8 else dt
    write = build_fused_rope_cache_module(head_dim=d, num_q_heads=qh, num_kv_heads=kh, block_size=bs,
                                          flash_layout=layout == "flash", dtype_str=dtype, apply_scale=fp8,
                                          reuse_freqs_front_part=reuse, pos_dtype="i64" if i64 else "i32")
    shapes = {"flash": ((nb, bs, kh, d),) * 2, "atom": ((nb, kh, d // 16, bs, 16), (nb, kh, d, bs)),
              "trans": ((nb, kh, d // 16, bs, 16), (nb, kh, bs // 16, d, 16))}[layout]
    scale = torch.tensor([0.02], device=DEV) if fp8 else None

    def call():
        kc, vc = (torch.zeros(s, dtype=cdt, device=DEV) for s in shapes)
        qo, ko = torch.empty(T, qh, d, dtype=dt, device=DEV), torch.empty(T, kh, d, dtype=dt, device=DEV)
        write(q, k, v, pos, cos, sin, slots, kc, vc, qo, ko, T, scale, scale)
        return kc, vc, qo, ko

    both(monkeypatch, call)


@pytest.mark.parametrize("quant,group,scale,weighted,three_d", [(True, 64, "fp32", False, False),
                                                                 (True, 128, "e8m0", True, True),
                                                                 (False, None, "fp32", True, True)])
def test_qknr_native_equals_python(quant, group, scale, weighted, three_d, monkeypatch):
    T, h, d, rd = 33, 3, 256, 64
    g = torch.Generator(device=DEV).manual_seed(5)
    rand = lambda *s: torch.randn(*s, generator=g, device=DEV).to(torch.bfloat16)
    q, kv, w, cos, sin = rand(T, h * d), strided(rand(T, d), (1,)), rand(d), rand(40, rd // 2), rand(40, rd // 2)
    q = strided(q.view(T, h, d), (0,)) if three_d else q
    pos = torch.randint(0, 40, (T,), generator=g, device=DEV)
    both(monkeypatch, lambda: flydsl_qk_norm_rope_quant(
        q, kv, w, cos, sin, pos, num_q_heads=h, head_dim=d, rope_head_dim=rd, q_weight=w if weighted else None,
        quant=quant, quant_group_size=group, scale_dtype=scale))


def test_mla_native_equals_python(monkeypatch):
    cfg = workloads.MlaConfig("x", 3, 700)
    x = workloads.build_mla_inputs(cfg, DEV)
    meta = [torch.empty(n, dtype=t, device=DEV) for n, t in get_mla_metadata_info_v1(3, 1, 128)]
    get_mla_metadata_v1(x["qo_indptr"], x["kv_indptr"], x["kv_last_page_lens"], 128, 1, True, meta[0], meta[2],
                        meta[1], meta[3], meta[4], meta[5])
    n = max(1, int(meta[0][2]))
    so, sl = torch.empty(n, 1, 128, 512, device=DEV), torch.empty(n, 1, 128, 1, device=DEV)

    def call():
        out = torch.zeros(3, 128, 512, dtype=torch.bfloat16, device=DEV)
        flydsl_mla_fwd_decode(x["q"], x["kvs"][0], x["kv_indices"], meta[1], meta[2], out, so, sl, 0.05)
        mla_reduce_v1(so, sl, meta[3], meta[4], meta[5], 1, out)
        return (out,)

    both(monkeypatch, call)


def test_forms_left_to_python():
    """Forms the native path does not take come back as None, unlaunched."""
    case = to_dev(make_case(batch=2, ctx=[40, 90], seed=3))
    out = torch.full(case["query"].shape, 5.0, dtype=torch.bfloat16, device=DEV)
    args = [out, case["query"], case["key_cache"], case["value_cache"], case["context_lengths"], None, None, 0.1,
            case["key_scale"], case["value_scale"], 0, None, case["block_tables"], 8, None, None, None, pd._plan,
            pd._native_workspace]
    changes = {1: case["query"].float(), 3: case["value_cache"].cpu(), 4: case["context_lengths"].long(), 7: 1,
               8: 0.5, 10: None, 12: None, 0: out.as_subclass(type("T", (torch.Tensor,), {})), 2: case["key_cache"].to(torch.bfloat16),
               14: torch.zeros(2, 2, 8, 4, device=DEV)}
    for i, x in changes.items():
        a = list(args)
        a[i] = x
        assert _lib.native().pa_decode(*a) is None, i
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        assert _lib.native().pa_decode(*args) is None  # under capture
    torch.cuda.synchronize()
    assert bool((out == 5.0).all())


def refused(call, args, changes):
    """Every single change of ``args`` comes back as None, unlaunched."""
    for i, x in changes:
        a = list(args)
        a[i] = x
        assert call(*a) is None, (i, x)


class Subclass(torch.Tensor):
    pass


def test_rope_forms_left_to_python():
    T, qh, kh, d, bs, nb = 5, 4, 2, 64, 16, 4
    bf = lambda *s: torch.ones(*s, dtype=torch.bfloat16, device=DEV)
    kc, vc = (torch.full(s, 7, dtype=torch.uint8, device=DEV) for s in ((nb, kh, d // 16, bs, 16), (nb, kh, d, bs)))
    qo, ko = bf(T, qh, d) * 5, bf(T, kh, d) * 5
    pos = torch.arange(T, dtype=torch.int32, device=DEV)
    one = torch.ones(1, device=DEV)
    args = [(d, qh, kh, bs, 0, 1, 1, 1, 0), bf(T, qh, d), bf(T, kh, d), bf(T, kh, d), pos, bf(9, d // 2), bf(9, d // 2),
            pos.clone(), kc, vc, qo, ko, T, one, one.clone()]
    refused(_lib.native().rope, args, [
        (1, bf(T, qh, 2 * d)[..., ::2]), (1, bf(T + 1, qh, d)), (1, bf(T, qh, d).half()), (1, bf(T, qh, d).as_subclass(Subclass)),
        (2, bf(T, kh, d).cpu()), (3, bf(T, kh + 1, d)), (4, pos.long()), (4, pos[:-1]), (5, bf(9, d)), (6, bf(8, d // 2)),
        (7, pos.view(1, -1)), (8, kc.to(torch.bfloat16)), (8, kc.transpose(0, 1)), (9, vc[:, :, :, :8]),
        (9, vc.view(nb, kh, 1, d, bs)[:-1]), (10, qo.half()), (11, bf(T, kh, d, 1)), (12, T - 1), (12, 0), (12, float(T)),
        (13, None), (13, one.double()), (14, one[:0])])
    assert bool((kc == 7).all()) and bool((vc == 7).all()) and bool((qo == 5).all()) and bool((ko == 5).all())


def test_qknr_forms_left_to_python():
    T, h, d, rd = 5, 2, 128, 64
    bf = lambda *s: torch.ones(*s, dtype=torch.bfloat16, device=DEV)
    pos = torch.zeros(T, dtype=torch.int64, device=DEV)
    args = [bf(T, h * d), bf(T, d), bf(d), bf(9, rd // 2), bf(9, rd // 2), pos, h, d, rd, None, True, 64, 0]
    refused(_lib.native().qknr, args, [
        (0, bf(T, h * d).half()), (0, bf(T, h * d + 1)[:, 1:]), (0, bf(T, d, h).transpose(1, 2)), (0, bf(0, h * d)),
        (0, bf(T, h * d).as_subclass(Subclass)), (1, bf(T - 1, d)), (1, bf(T, d + 1)[:, :d]), (1, bf(T, d).cpu()), (2, bf(d + 1)),
        (2, bf(2 * d)[::2]), (3, bf(9, rd)), (4, bf(8, rd // 2)), (4, bf(9, rd // 2).float()), (5, pos.int()), (5, pos[:-1]),
        (6, h + 1), (9, bf(d).float()), (9, bf(d - 1)), (11, 48), (11, 0)])


def test_mla_forms_left_to_python():
    fp8 = lambda *s: torch.zeros(*s, dtype=torch.uint8, device=DEV).view(torch.float8_e4m3fn)
    i32 = lambda *s: torch.zeros(*s, dtype=torch.int32, device=DEV)
    R, n = 2, 3
    out = torch.full((R, 128, 512), 5.0, dtype=torch.bfloat16, device=DEV)
    so, sl = torch.zeros(n, 1, 128, 512, device=DEV), torch.zeros(n, 1, 128, 1, device=DEV)
    args = [fp8(R, 128, 576), fp8(9, 1, 1, 576), i32(9), i32(3), i32(2, 8), out, so, sl, 0.05, False]
    refused(_lib.native().mla_decode, args, [
        (0, fp8(R, 64, 576)), (0, fp8(R, 128, 576).view(torch.uint8)), (0, fp8(R, 128, 576).view(torch.float8_e4m3fnuz)),
        (0, fp8(0, 128, 576)), (1, fp8(9, 2, 1, 576)), (1, fp8(9, 1, 576)), (1, fp8(9, 1, 1, 576).cpu()), (2, i32(9).long()),
        (2, i32(18)[::2]), (3, i32(0)), (4, i32(2, 8).float()), (5, out.float()), (5, out[:1]), (5, out.transpose(0, 1)),
        (6, so.half()), (6, so[:2]), (7, sl[..., 0]), (8, 1), (0, fp8(R, 128, 576).as_subclass(Subclass))])
    args = [so, sl, i32(R + 1), i32(R, 2), i32(n), out]
    refused(_lib.native().mla_reduce, args, [
        (0, so.double()), (0, so.transpose(0, 2)), (1, sl.cpu()), (2, i32(R + 1).long()), (2, i32(0)), (2, i32(R + 2)),
        (3, i32(R, 4)[:, ::2]), (4, i32(n).short()), (5, out.half()), (5, out[..., :256].contiguous()),
        (5, out.transpose(0, 1))])
    torch.cuda.synchronize()
    assert bool((out == 5.0).all())
