"""Portions cut into segments of single chunks against the token-by-token recurrence: lengths around the chunks' edges (16 tokens; cut from the
third chunk on), ragged sequences with and without an earlier state, so many sequences that segments get longer, and workspaces that
hold only the coarse segments of 8 chunks, or not even these; fixed decays, whose segments never get shorter."""
import ctypes
import os

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def amd():
    import light_vllm_amd._custom_ops  # noqa: F401
    return torch.ops._C_amd


def operands(lengths, heads, dk, dv, bonus, seed=0):
    g = torch.Generator().manual_seed(seed)
    rows, n, rank = sum(lengths), len(lengths), 24
    r = lambda *s: torch.randn(*s, generator=g)
    t = {"q": r(rows, heads * dk), "k": r(rows, heads * dk), "v": r(rows, heads * dv), "u": r(rows, rank), "gate": r(rows, heads * dv)}
    t = {k: v.bfloat16().to(DEV) for k, v in t.items()}
    t["a_t"], t["bias"] = (0.3 * r(rank, heads * dk)).to(DEV), r(heads * dk).to(DEV)
    t["bonus"] = r(heads * dk).to(DEV) if bonus else None
    t["weight"] = r(heads * dv).to(DEV)
    t["state"] = r(n + 1, heads, dk, dv).to(DEV)
    t["slots"] = torch.arange(n, 0, -1, dtype=torch.int32, device=DEV)
    t["start"] = torch.tensor([0] + lengths).cumsum(0).int().to(DEV)
    t["lens"] = torch.tensor([m + (7 if i % 2 else 0) for i, m in enumerate(lengths)], dtype=torch.int32, device=DEV)  # odd ones go on
    return t


def reference(amd, t, kind, inv_tau, scale):
    state = t["state"].clone()
    decay = amd.log_decay(t["u"], t["a_t"], t["bias"], kind, inv_tau)
    o = amd.recurrent_scan(t["q"], t["k"], t["v"], decay, t["bonus"], scale, state, t["slots"], t["start"], t["lens"])
    out = torch.empty_like(t["v"])
    amd.head_norm_gate(out, o, t["gate"], t["weight"], 1e-5, 1.0)
    return out, state


def check(out, state, want, want_state):
    # both sides: fp32 sums of up to some hundred products, then one rounding to bf16 (2^-8 of the value between neighbours)
    torch.testing.assert_close(state, want_state, rtol=2e-4, atol=2e-4 * float(want_state.abs().max()))
    torch.testing.assert_close(out.float(), want.float(), rtol=2 ** -7, atol=2 ** -9 * float(want.float().abs().max()))


@pytest.mark.parametrize("heads,dk,dv,kind,bonus", [(8, 128, 128, 0, False), (32, 64, 64, 1, True), (2, 48, 136, 0, False)])
@pytest.mark.parametrize("lengths", [[32], [33], [47, 1, 48, 49], [65, 16, 17, 2], [300], [128, 129, 127], [40] + [1] * 400],
                         ids=lambda v: "-".join(map(str, v[:4])))
def test_segments(amd, lengths, heads, dk, dv, kind, bonus):
    t = operands(lengths, heads, dk, dv, bonus)
    inv_tau, scale = (1 / 16, dk ** -0.5) if kind == 0 else (1.0, 1.0)
    want, want_state = reference(amd, t, kind, inv_tau, scale)
    out, state = torch.empty_like(t["v"]), t["state"].clone()
    amd.recurrent_mix(out, t["q"], t["k"], t["v"], t["u"], t["a_t"], t["bias"], kind, inv_tau, t["bonus"], scale, t["gate"], t["weight"],
                      1e-5, 1.0, state, t["slots"], t["start"], t["lens"], max(lengths))
    check(out, state, want, want_state)


@pytest.mark.parametrize("heads,dk,dv", [(3, 64, 64), (2, 128, 30)])
@pytest.mark.parametrize("lengths", [[80], [81], [64, 65, 80, 81, 96, 97]], ids=lambda v: "-".join(map(str, v)))
def test_few_segments_and_more(amd, lengths, heads, dk, dv):
    """Up to five segments of a sequence are asked for four at a time, more of them sixteen at a time; columns in fours and one by one."""
    test_segments(amd, lengths, heads, dk, dv, 0, False)


@pytest.mark.parametrize("lengths", [[1] * 20 + [33] + [1] * 3 + [16, 17, 49] + [1] * 9, [3, 64, 1, 1, 65, 2, 15, 48], [1] * 255 + [45], [45] + [1] * 255])
def test_single_tokens_beside_segments(amd, lengths):
    test_segments(amd, lengths, 8, 64, 64, 0, False)


def test_smaller_workspaces(amd):
    import light_vllm_amd
    lib = ctypes.CDLL(os.path.join(os.path.dirname(light_vllm_amd.__file__), "lib", "liblvllm_hybrid.so"))
    lib.lvllm_recurrent_mix_workspace_bytes.restype = ctypes.c_int64
    heads, dk, dv, lengths, scale = 8, 64, 64, [300, 77], 64 ** -0.5
    t = operands(lengths, heads, dk, dv, False)
    rows = sum(lengths)
    most = lib.lvllm_recurrent_mix_workspace_bytes(rows, 2, heads, dk, dv, max(lengths))
    # decays, and of segments of 128 rows a state and a decay for each: rows / 128 + sequences + 1
    coarse = 4 * (rows * heads * dk + (rows // 128 + 3) * heads * (dk * dv + 64))
    assert most > coarse
    want, want_state = reference(amd, t, 0, 1 / 16, scale)
    f, i, i64, p = ctypes.c_float, ctypes.c_int, ctypes.c_int64, lambda x: ctypes.c_void_p(0 if x is None else x.data_ptr())
    for room, code in ((most, 0), (most - 4, 0), (coarse, 0), (coarse - 4, 1)):
        out, state = torch.zeros_like(t["v"]), t["state"].clone()
        ws = torch.empty(most, dtype=torch.uint8, device=DEV)
        ws[room:] = 77
        rc = lib.lvllm_recurrent_mix(
            p(out), i64(out.stride(0)), p(t["q"]), p(t["k"]), p(t["v"]), i64(heads * dk), i64(heads * dk), i64(heads * dv), p(t["u"]),
            i64(t["u"].stride(0)), p(t["a_t"]), p(t["bias"]), i(t["u"].shape[1]), i(0), f(1 / 16), p(None), f(scale), p(t["gate"]),
            i64(heads * dv), p(t["weight"]), i(dv), f(1e-5), f(1.0), p(state), i64(state.stride(0)), p(t["slots"]), i(state.shape[0]),
            p(t["start"]), p(t["lens"]), i(2), i(rows), i(heads), i(dk), i(dv), i(max(lengths)), p(ws), i64(room), i(DTYPE_BF16),
            ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        assert (rc != 0) == (code != 0), (room, rc)
        torch.cuda.synchronize()
        assert bool((ws[room:] == 77).all())
        if code == 0:
            check(out, state, want, want_state)


def test_retention_of_any_workspace(amd):
    """A retention's bits do not depend on how much scratch there is."""
    import light_vllm_amd
    lib = ctypes.CDLL(os.path.join(os.path.dirname(light_vllm_amd.__file__), "lib", "liblvllm_local.so"))
    heads, dk, dv, lengths = 8, 64, 64, [300, 77, 1]
    t, rows, n, results = operands(lengths, heads, dk, dv, False), sum(lengths), len(lengths), []
    decay = torch.linspace(0.9, 0.999, heads, dtype=torch.float64)
    decay = torch.stack([decay, decay.log()]).float().to(DEV)
    positions = torch.cat([torch.arange(m) + (7 if i % 2 else 0) for i, m in enumerate(lengths)]).to(DEV)
    turns = torch.tensor([0.1, 0.01], dtype=torch.float64, device=DEV)
    # rotated queries and keys, and of segments of 128 rows a state and a decay for each: rows / 128 + sequences + 1
    least = 4 * (2 * rows * heads * dk + (rows // 128 + n + 1) * heads * (dk * dv + 64))
    f, i, i64, p = ctypes.c_float, ctypes.c_int, ctypes.c_int64, lambda x: ctypes.c_void_p(0 if x is None else x.data_ptr())
    for room in (least, 8 * least):
        out, state, ws = torch.zeros_like(t["v"]), t["state"].clone(), torch.empty(room, dtype=torch.uint8, device=DEV)
        rc = lib.lvllm_retention(
            p(out), i64(out.stride(0)), p(t["q"]), p(t["k"]), p(t["v"]), i64(heads * dk), i64(heads * dk), i64(heads * dv), p(positions),
            p(turns), i(4), p(decay), f(dk ** -0.5), p(t["gate"]), i64(heads * dv), p(t["weight"]), i(dv), f(1e-5), f(1.0), p(state),
            i64(state.stride(0)), p(t["slots"]), i(state.shape[0]), p(t["start"]), p(t["lens"]), i(n), i(rows), i(heads), i(dk), i(dv),
            i(max(lengths)), p(ws), i64(room), i(DTYPE_BF16), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        assert rc == 0
        torch.cuda.synchronize()
        results.append((out, state))
    (a, sa), (b, sb) = results
    assert bool(a.any(1).all()) and torch.equal(a, b) and torch.equal(sa, sb)


@pytest.mark.parametrize("heads,dk,dv", [(8, 128, 128), (3, 128, 120), (2, 48, 24), (2, 256, 64), (4, 64, 36), (2, 64, 130)])
@pytest.mark.parametrize("lengths", [[300], [49], [48], [65, 1, 200]], ids=lambda v: "-".join(map(str, v)))
def test_retention_of_narrow_slices(amd, heads, dk, dv, lengths):
    """Columns cut finer, with a norm behind, where there is scratch for the read-outs: the same bits as without it."""
    import light_vllm_amd
    lib = ctypes.CDLL(os.path.join(os.path.dirname(light_vllm_amd.__file__), "lib", "liblvllm_local.so"))
    lib.lvllm_retention_workspace_bytes.restype = ctypes.c_int64
    t, rows, n, results = operands(lengths, heads, dk, dv, False), sum(lengths), len(lengths), []
    decay = torch.linspace(0.9, 0.999, heads, dtype=torch.float64)
    decay = torch.stack([decay, decay.log()]).float().to(DEV)
    positions = torch.cat([torch.arange(m) + (7 if i % 2 else 0) for i, m in enumerate(lengths)]).to(DEV)
    turns = torch.tensor([0.1, 0.01], dtype=torch.float64, device=DEV)
    most = lib.lvllm_retention_workspace_bytes(rows, n, heads, dk, dv, max(lengths))
    f, i, i64, p = ctypes.c_float, ctypes.c_int, ctypes.c_int64, lambda x: ctypes.c_void_p(0 if x is None else x.data_ptr())
    for room in ((most, most - 4) if dv <= 128 and max(lengths) > 48 else (most,)):
        out, state, ws = torch.zeros_like(t["v"]), t["state"].clone(), torch.empty(most, dtype=torch.uint8, device=DEV)
        ws[room:] = 77
        rc = lib.lvllm_retention(
            p(out), i64(out.stride(0)), p(t["q"]), p(t["k"]), p(t["v"]), i64(heads * dk), i64(heads * dk), i64(heads * dv), p(positions),
            p(turns), i(4), p(decay), f(dk ** -0.5), p(t["gate"]), i64(heads * dv), p(t["weight"]), i(dv), f(1e-5), f(1.0), p(state),
            i64(state.stride(0)), p(t["slots"]), i(state.shape[0]), p(t["start"]), p(t["lens"]), i(n), i(rows), i(heads), i(dk), i(dv),
            i(max(lengths)), p(ws), i64(room), i(DTYPE_BF16), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        assert rc == 0
        torch.cuda.synchronize()
        assert bool((ws[room:] == 77).all())
        results.append((out, state))
    for a, sa in results:
        assert bool(a.any(1).all()) and torch.equal(a, results[0][0]) and torch.equal(sa, results[0][1])
    # against the token-by-token recurrence: fp32 sums of rotated values, one rounding to bf16
    decays = decay[1].repeat_interleave(dk).expand(rows, -1).contiguous()
    angles = 2 * torch.pi * positions[:, None].double() * turns

    def rotated(x):
        x = x.float().view(rows, heads, dk).clone()
        c, s = angles.cos().float()[:, None], angles.sin().float()[:, None]
        u, w = x[..., :2].clone(), x[..., 2:4].clone()
        x[..., :2], x[..., 2:4] = u * c - w * s, w * c + u * s
        return x.reshape(rows, heads * dk)
    want_state, g = t["state"].clone(), t["gate"].float()
    o = amd.recurrent_scan(rotated(t["q"]), rotated(t["k"]), t["v"].float(), decays, None, dk ** -0.5, want_state, t["slots"], t["start"],
                           t["lens"])
    want = torch.empty_like(g)
    amd.head_norm_gate(want, o, g, t["weight"], 1e-5, 1.0)
    check(results[0][0], results[0][1], want, want_state)


DTYPE_BF16 = 2
