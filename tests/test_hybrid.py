"""Purusun on the host: the plain implementation (oracle/purusun.py) against closed forms and torch's own functions, the registry
and the checkpoint reader, the packed weights, the cache's shapes and the dense library's argument checks."""

import ctypes
import json
import math

import pytest
import torch
from safetensors.torch import save_file

from ajllm_amd import _lib, checkpoint, dense, hybrid, modeling
from oracle import purusun as O
from tests.hybrid_models import SCALING, attention, config, random_weights, scan

F = torch.nn.functional


# ------------------------------------------------------------------ the plain implementation
def test_norms_and_activations_match_torch():
    x, w = torch.randn(5, 12, dtype=torch.float64), torch.randn(12, dtype=torch.float64)
    assert torch.allclose(O.centered_rms_norm(x, w, 1e-3), F.rms_norm(x, (12,), 1 + w, 1e-3))
    norm = modeling.build_norm("zero_centered_rmsnorm", 12, 1e-3)
    assert (norm.weight == 0).all()
    with torch.no_grad():
        norm.weight.copy_(w)
        assert torch.allclose(norm(x.float()), F.rms_norm(x.float(), (12,), 1 + w.float(), 1e-3), atol=1e-5)
    z = torch.cat((torch.linspace(-60, 60, 41, dtype=torch.float64), torch.zeros(1, dtype=torch.float64)))
    assert torch.allclose(O.softplus(z), F.softplus(z, threshold=1000)) and torch.allclose(O.silu(z), F.silu(z))
    h, up, down = torch.randn(3, 6), torch.randn(10, 6), torch.randn(6, 10)
    ff = modeling.build_feed_forward("squared_relu", 6, 10)
    with torch.no_grad():
        ff.w1.weight.copy_(up)
        ff.w2.weight.copy_(down)
        assert torch.allclose(ff(h), O.squared_relu(h, up, down), atol=1e-5)


def test_frequency_scaling_keeps_blends_and_divides():
    dims, base = 64, 500.0
    plain = [O.frequency(base, dims, i, None) for i in range(dims // 2)]
    scaled = [O.frequency(base, dims, i, SCALING) for i in range(dims // 2)]
    kinds = set()
    for f, s in zip(plain, scaled):
        wavelength = 2 * math.pi / f
        if wavelength < SCALING["original"] / SCALING["high"]:
            kinds.add("kept")
            assert s == f
        elif wavelength > SCALING["original"] / SCALING["low"]:
            kinds.add("divided")
            assert s == f / SCALING["factor"]
        else:
            kinds.add("between")
            assert f / SCALING["factor"] <= s <= f
    assert kinds == {"kept", "between", "divided"}
    assert all(a >= b for a, b in zip(scaled, scaled[1:]))   # the blend meets both ends: no jump upwards
    for scaling in (None, SCALING):
        held = dense.FrequencyScaling(**{k: float(v) for k, v in scaling.items()}) if scaling else None
        got = dense.rotary_frequencies(base, dims, held)
        want = torch.tensor([O.frequency(base, dims, i, scaling) for i in range(dims // 2)], dtype=torch.float64)
        assert torch.allclose(got, want, rtol=1e-14, atol=0)


def test_rotation_turns_halves_and_is_relative():
    rot = {"dims": 8, "base": 50.0, "scaling": None}
    v = torch.randn(11, dtype=torch.float64)
    out = O.rotate(v, 9, rot)
    for i in range(4):
        turned = torch.view_as_complex(torch.stack((v[i], v[i + 4]))) * torch.polar(torch.tensor(1.0).double(), torch.tensor(9 * 50.0 ** (-i / 4)).double())
        assert torch.allclose(torch.view_as_real(turned), torch.stack((out[i], out[i + 4])))
    assert torch.equal(out[8:], v[8:])
    a, b = torch.randn(8, dtype=torch.float64), torch.randn(8, dtype=torch.float64)
    assert torch.allclose(O.rotate(a, 5, rot) @ O.rotate(b, 3, rot), O.rotate(a, 2005, rot) @ O.rotate(b, 2003, rot))


def test_window_beside_kept_first_tokens():
    for window, keep in ((4, 0), (4, 2), (1, 1), (3, 9), (None, 0)):
        mask = O.visible_mask(12, window, keep)
        for i in range(12):
            near = range(0 if window is None else max(0, i - window + 1), i + 1)
            want = sorted(set(near) | set(range(min(keep, i + 1))))
            assert [j for j in range(12) if mask[i, j]] == want == [j for j in range(12) if O.visible(i, j, window, keep)]


def test_attention_is_torchs_with_keys_as_values():
    spec = attention(heads=6, kv_heads=2, dim=10, rot=4, window=5, keep=2)
    w = {k[len("l0.mix."):]: v.double() for k, v in random_weights(config([spec], loop=None), 3).items() if k.startswith("l0.mix.")}
    h = torch.randn(20, 48, dtype=torch.float64)
    raw = (h @ w["k"].T).view(20, 2, 10)
    q = O.rotate_rows(F.rms_norm((h @ w["q"].T).view(20, 6, 10), (10,), w["q.norm"], 1e-5), spec["mixer"]["rot"])
    k = O.rotate_rows(F.rms_norm(raw, (10,), w["k.norm"], 1e-5), spec["mixer"]["rot"])
    got = F.scaled_dot_product_attention(q.transpose(0, 1), k.transpose(0, 1).repeat_interleave(3, 0), raw.transpose(0, 1).repeat_interleave(3, 0),
                                         attn_mask=O.visible_mask(20, 5, 2), scale=spec["mixer"]["scale"])
    want = (got.transpose(0, 1).reshape(20, 60) * torch.sigmoid(h @ w["g"].T)) @ w["o"].T
    assert torch.allclose(O.key_value_attention(h, w, spec["mixer"], 1e-5), want)


def test_convolution_is_torchs():
    x, w, b = torch.randn(9, 5, dtype=torch.float64), torch.randn(5, 4, dtype=torch.float64), torch.randn(5, dtype=torch.float64)
    want = F.conv1d(F.pad(x.T[None], (3, 0)), w[:, None], b, groups=5)[0].T
    assert torch.allclose(O.causal_conv(x, w, b), want)


def test_recurrence_in_closed_form_and_from_a_state():
    t, ch, n = 7, 3, 2
    x, dt = torch.randn(t, ch, dtype=torch.float64), torch.rand(t, ch, dtype=torch.float64)
    a, d = -torch.rand(ch, n, dtype=torch.float64), torch.randn(ch, dtype=torch.float64)
    b, c = torch.randn(t, n, dtype=torch.float64), torch.randn(t, n, dtype=torch.float64)
    y, last = O.recurrence(x, dt, a, b, c, d)
    for i in range(t):
        for k in range(ch):
            want = float(d[k] * x[i, k])
            for j in range(i + 1):
                for m in range(n):
                    decay = math.exp(float(a[k, m]) * float(dt[j + 1:i + 1, k].sum()))
                    want += decay * float(dt[j, k] * x[j, k] * b[j, m] * c[i, m])
            assert float(y[i, k]) == pytest.approx(want)
    head, state = O.recurrence(x[:3], dt[:3], a, b[:3], c[:3], d)
    tail, end = O.recurrence(x[3:], dt[3:], a, b[3:], c[3:], d, state)
    assert torch.allclose(torch.cat((head, tail)), y) and torch.allclose(end, last)


def test_hyper_connection_reads_mixes_and_writes():
    """One stream with neutral coefficients is the plain residual sum; the mix is indexed [from, to], all from the old streams."""
    x = torch.randn(1, 4, 6, dtype=torch.float64)
    one = {"in": torch.ones(1).double(), "out": torch.ones(1).double(), "mix": torch.ones(1, 1).double()}
    assert torch.allclose(O.hyper_sublayer(x, one, torch.sin), x + torch.sin(x))
    x = torch.randn(2, 4, 6, dtype=torch.float64)
    hc = {"in": torch.tensor([2.0, -1.0]).double(), "out": torch.tensor([0.5, 3.0]).double(), "mix": torch.tensor([[1.0, 10.0], [0.0, 1.0]]).double()}
    got = O.hyper_sublayer(x, hc, torch.sin)
    y = torch.sin(2 * x[0] - x[1])
    assert torch.allclose(got[0], x[0] + 0.5 * y) and torch.allclose(got[1], 10 * x[0] + x[1] + 3 * y)


def test_loop_order():
    assert O.layer_order(4, {"start": 1, "stop": 3, "times": 2}) == [0, 1, 2, 1, 2, 3]
    assert O.layer_order(2, None) == [0, 1] and O.layer_order(2, {"start": 0, "stop": 2, "times": 1}) == [0, 1]


def test_later_tokens_do_not_change_earlier_logits():
    cfg = config()
    w = random_weights(cfg, 3)
    tokens = list(range(14))
    full = O.forward(cfg, w, tokens)
    assert torch.allclose(O.forward(cfg, w, tokens[:8]), full[:8])
    other = O.forward(cfg, w, [5] + tokens[1:])
    assert not torch.allclose(other[-1], full[-1])


# ------------------------------------------------------------------ registry, configuration, weights
def test_registry_builds_the_architecture_and_refuses_others():
    cfg = config()
    with torch.device("meta"):
        model = modeling.build_model(cfg)
    assert isinstance(model, hybrid.HybridLM) and [i for i, _ in model.runs] == O.layer_order(4, cfg["loop"])
    assert set(model.checkpoint_names().values()) == set(random_weights(cfg, 0))
    bare = attention(window=None)
    bare["mixer"].update(rot=None, mask=None)
    with torch.device("meta"):
        mix = modeling.build_model(config([bare], loop=None)).layers[0].mixer
    assert mix.window is None and mix.rot_dim == 0
    for change, message in (({"type": "other"}, "mixer"), ({"mlp": {"kind": "sparse", "ff": 8}}, "feed-forward")):
        with pytest.raises(ValueError, match=message):
            modeling.build_model(config([{**scan(), **change}], loop=None))
    for bad, message in ((attention(heads=5, kv_heads=2), "divisible"), (attention(rot=18), "rotated"), (attention(rot=7), "rotated")):
        with pytest.raises(ValueError, match=message):
            modeling.build_model(config([bad], loop=None))
    odd = attention()
    odd["mixer"]["vdim"] = 8
    with pytest.raises(ValueError, match="vdim"):
        modeling.build_model(config([odd], loop=None))
    with pytest.raises(ValueError, match="loop"):
        modeling.build_model(config(loop={"start": 2, "stop": 9, "times": 2}))


def _folder(tmp_path, cfg, weights):
    (tmp_path / "config.json").write_text(json.dumps(cfg))
    save_file({k: v.to(torch.bfloat16).contiguous() for k, v in weights.items()}, str(tmp_path / "model.safetensors"))
    return tmp_path


def test_checkpoint_folder_loads_strictly(tmp_path):
    cfg = config([scan(ff=None), attention()], loop=None)
    w = random_weights(cfg, 1)
    model = checkpoint.load_model(_folder(tmp_path, cfg, w), "cpu", torch.float32)
    state = model.state_dict()
    for key, name in model.checkpoint_names().items():
        assert torch.equal(state[key], w[name])
    assert model.layers[0].feed_forward is None and model.layers[0].hyper2 is None
    extra = {**w, "l0.norm2": torch.ones(cfg["width"]), "l0.hc2.in": torch.ones(3)}   # of a sublayer that is not there
    checkpoint.load_model(_folder(tmp_path, cfg, extra), "cpu")
    with pytest.raises(ValueError, match="unexpected"):
        checkpoint.load_model(_folder(tmp_path, cfg, {**w, "l1.mix.v": torch.ones(3)}), "cpu")
    with pytest.raises(ValueError, match="missing"):
        checkpoint.load_model(_folder(tmp_path, cfg, {k: v for k, v in w.items() if k != "l0.mix.D"}), "cpu")


def test_the_model_has_no_cpu_path(tmp_path):
    cfg = config()
    model = checkpoint.load_model(_folder(tmp_path, cfg, random_weights(cfg, 1)), "cpu")
    with pytest.raises(ValueError, match="ROCm"):
        model(torch.zeros((1, 3), dtype=torch.long))


def test_packed_attention_computes_the_same_projections():
    cfg = config([attention(heads=3, kv_heads=1, dim=12, rot=6)], width=52, loop=None)
    model = modeling.build_model(cfg)
    mix = model.layers[0].mixer
    with torch.no_grad():
        for p in model.parameters():
            p.normal_()
        w = hybrid.PackedAttention(mix, 64)
        h, joined = torch.randn(52), torch.randn(3, 12)
        y = w.w_in @ F.pad(h, (0, 12))
        parts = y.view(7, 16)
        want = torch.cat((mix.q_proj.weight, mix.k_proj.weight, mix.gate_proj.weight)) @ h
        assert torch.allclose(parts[:, :12].reshape(-1), want, atol=1e-4) and (parts[:, 12:] == 0).all()
        assert torch.allclose(y[w.gate_column:].view(3, 16)[:, :12].reshape(-1), mix.gate_proj.weight @ h, atol=1e-4)
        out = w.w_out @ F.pad(joined, (0, 4)).reshape(-1)
        assert torch.allclose(out[:52], mix.output_proj.weight @ joined.reshape(-1), atol=1e-4) and (out[52:] == 0).all()
        assert torch.equal(w.q_gain[:12], mix.q_norm.weight) and (w.q_gain[12:] == 0).all()
        assert torch.allclose(w.half_turns * math.pi, dense.rotary_frequencies(300.0, 6), rtol=1e-15)


def test_packed_scan_computes_the_same_projections():
    cfg = config([scan(inner=20, state=5, rank=3, conv=2)], width=44, loop=None)
    model = modeling.build_model(cfg)
    mix = model.layers[0].mixer
    with torch.no_grad():
        for p in model.parameters():
            p.normal_()
        w = hybrid.PackedScan(mix, 48)
        assert (w.inner, w.states, w.rank, w.taps, w.low_rows) == (32, 8, 8, 2, 32)
        h, x, dt = torch.randn(44), torch.randn(20), torch.randn(3)
        y = (w.w_in @ F.pad(h, (0, 4))).view(2, 32)
        assert torch.allclose(y[:, :20].reshape(-1), mix.in_proj.weight @ h, atol=1e-4) and (y[:, 20:] == 0).all()
        low, want = w.w_low @ F.pad(x, (0, 12)), mix.x_proj.weight @ x
        assert torch.allclose(low[:3], want[:3], atol=1e-4) and torch.allclose(low[8:13], want[3:8], atol=1e-4)
        assert torch.allclose(low[16:21], want[8:], atol=1e-4) and (low[[3, 7, 13, 15, 21]] == 0).all()
        assert torch.allclose((w.w_dt @ F.pad(dt, (0, 5)))[:20], mix.dt_proj.weight @ dt, atol=1e-5)
        planes = w.a2.permute(1, 0, 2).reshape(32, 8)    # [channels, states]
        assert torch.allclose(planes[:20, :5] * math.log(2), -torch.exp(mix.a_log), rtol=1e-6) and (planes[20:] == 0).all() and (planes[:, 5:] == 0).all()
        assert torch.equal(w.conv[1, :20], mix.conv_weight[:, 1])   # the last row meets the token itself


def test_cache_holds_windows_kept_rows_columns_and_states():
    cfg = config([attention(window=5, keep=2), attention(window=9, keep=0), attention(window=None), scan(conv=1, state=6), scan(inner=20)],
                 loop={"start": 0, "stop": 1, "times": 2})
    model = modeling.build_model(cfg)
    cache = model.new_cache(2, 8)
    assert [tuple(r.shape) for r in cache.rings] == [(2, 2, 7, 32), (2, 2, 7, 32), (2, 2, 8, 32), (2, 2, 8, 32), (2, 0, 48), (2, 3, 32)]
    assert cache.kept == [2, 2, 0, 0, 0, 0]
    assert [None if s is None else tuple(s.shape) for s in cache.states] == [None] * 4 + [(2, 2, 48, 4), (2, 2, 32, 4)]
    assert all(s.dtype == torch.float32 for s in cache.states[4:])
    part = cache.rows(1, 2)
    assert part.rings[0].data_ptr() == cache.rings[0][1].data_ptr() and part.states[4].data_ptr() == cache.states[4][1].data_ptr()
    with pytest.raises(ValueError, match="max_len"):
        model.new_cache(1)
    with pytest.raises(ValueError):
        model.new_cache(1, 8, torch.float16)


# ------------------------------------------------------------------ the library
def test_dense_library_refuses_bad_arguments_before_any_launch():
    lib = _lib.load_dense()
    buf = ctypes.create_string_buffer(4096)
    p = ctypes.c_void_p((ctypes.addressof(buf) + 15) & ~15)
    assert lib.ajqd_embed_streams(p, 1, p, 4, p, p, p, 17, 16, 0, None) == -4                            # streams
    assert lib.ajqd_streams_norm(p, p, None, None, None, p, p, 1e-5, p, None, 2, 1, 16, 16, 0, None) == -1
    assert lib.ajqd_streams_norm(p, None, None, None, None, p, p, 1e-5, p, None, 2, 1, 24, 16, 0, None) == -2
    assert lib.ajqd_dense_out_streams(p, p, p, p, p, p, None, p, 2, 1, 12, 16, None) == -2
    assert lib.ajqd_activation(p, p, 12, 0, 0, None) == -2 and lib.ajqd_activation(p, p, 16, 9, 0, None) == -4
    split = _lib.KeyValueSplitArgs(y=p, q_gain=p, k_gain=p, half_turns=p, q=p, rows=p, tokens=4, seq=4, ldy=48, heads=1, groups=1, dim=16, dimp=16,
                                   rot=18, q_ld=16, rows_batch=128, rows_head=128)
    assert lib.ajqd_key_value_split(ctypes.byref(split), 0, 0, None) == -2                               # rotates more than a head has
    split.rot, split.groups, split.rows_head = 8, 2, 64
    assert lib.ajqd_key_value_split(ctypes.byref(split), 0, 0, None) == -2 and b"overlap" in lib.ajqd_last_error()
    split.pos, split.cap, split.kept = p, 4, 4
    assert lib.ajqd_key_value_split(ctypes.byref(split), 0, 0, None) == -2                               # no slot beside the kept ones
    assert lib.ajqd_ring_copy(p, 6, 2, p, 8, 32, 0, 2, 5, 32, 1, 1, None) == -2                          # 5 positions for 4 moving slots
    assert lib.ajqd_group_merge(p, None, 0, p, 16, 1, 1, 1, 40, 16, None) == -2
    assert lib.ajqd_conv_silu(p, 16, None, p, p, 3, None, 2, 2, 16, 4, p, 0, None) == -1                 # no columns from before
    args = _lib.ScanArgs(x=p, dt=p, low=p, z=p, a2=p, d=p, dt_bias=p, out=p, batch=1, seq=2, inner=16, states=6, dt_ld=16, low_ld=16, z_ld=16, out_ld=16)
    assert lib.ajqd_scan(ctypes.byref(args), 0, None) == -2
    args.states, args.low_ld, args.start = 4, 16, 5
    assert lib.ajqd_scan(ctypes.byref(args), 0, None) == -1                                              # no state to start from
    args.start, args.states, args.low_ld, args.c_col = 0, 260, 600, 260
    assert lib.ajqd_scan(ctypes.byref(args), 0, None) == -4
    assert lib.ajqd_scan_project(p, 16, p, p, p, p, p, p, 1, 16, 4, 16, 1, None) == -2                   # y holds both halves
    step = _lib.ScanStepArgs(y=p, ring=p, weight=p, bias=p, pos=p, partial=p, w_dt=p, dt_bias=p, a2=p, d=p, state=p, out=p, batch=1, ldy=32, inner=16,
                             taps=4, rows=16, splits=1, rank=8, states=8, out_ld=16)
    assert lib.ajqd_scan_step(ctypes.byref(step), None) == -2                                            # 8 + 16 rows in 16


def test_every_form_of_a_decode_step_of_the_scan_is_run():
    from tests.test_gpu_hybrid import SCAN_FORMS, SCAN_LINES, STEPS
    lib, up = _lib.load_dense(), lambda n: -(-n // 16) * 16
    form = lambda batch, inner, states, rank, taps: (lib.ajqd_scan_form(batch, inner, up(rank + 2 * states), lib.ajqd_scan_splits(batch, inner), rank, states), taps == 4)
    got = {form(*s) for s in STEPS + SCAN_LINES + SCAN_FORMS}
    assert {(f // 100, four) for f, four in got} == {(10 * kb + rt, four) for kb in (2, 4, 8) for rt in (1, 2) for four in (True, False)}
    assert {f % 10 for f, _ in got} == {0, 4, 8} and {f // 10 % 10 for f, _ in got if f // 100 % 10 == 2} == {0, 1}


@pytest.mark.parametrize("batch,inner,rank,states,splits,sequences", [
    # the step: 16 channels, four sequences, eight in one round where four take two, and past two rounds of fours with up to 32 states
    (4, 4096, 128, 16, 16, 0), (5, 4096, 128, 16, 16, 4), (24, 8192, 256, 16, 16, 4), (13, 13440, 208, 16, 8, 8), (32, 8192, 256, 64, 8, 8), (16, 17360, 272, 16, 8, 4),
    (13, 18576, 512, 64, 8, 4), (31, 13440, 512, 16, 8, 8), (31, 13440, 512, 32, 8, 8), (48, 9712, 304, 36, 10, 4), (64, 12288, 384, 64, 8, 4),
    # parts of the projection, few sequences past 4096 channels
    (4, 4112, 256, 16, 9, 4), (5, 4112, 256, 16, 17, 4), (1, 5120, 160, 16, 10, 4), (1, 5136, 160, 16, 6, 4), (33, 4096, 128, 16, 8, 4),
])
def test_forms_of_a_decode_step_of_the_scan(batch, inner, rank, states, splits, sequences):
    lib = _lib.load_dense()
    assert lib.ajqd_scan_splits(batch, inner) == splits
    assert lib.ajqd_scan_form(batch, inner, -(-(rank + 2 * states) // 16) * 16, splits, rank, states) % 10 == sequences


def test_every_form_of_a_decode_product_is_run():
    """The shapes that the GPU test runs reach every form of a product without many streams that the library holds."""
    from tests.test_gpu_hybrid import FORMS
    lib = _lib.load_dense()
    forms = {lib.ajqd_dense_out_form(batch, k, width, 2, 0) for batch, k, width in FORMS}
    assert forms == {221110, 811110, 811111, 811112, 811114, 811210, 811214, 421110, 421111, 421121, 421112, 421122, 421114, 421124, 421210, 421214, 421220,
                     422210, 422214}
    assert forms >= {lib.ajqd_dense_out_form(b, k, 16 * n, s, 0) for b in (1, 3, 5, 8, 9, 17, 33, 64) for k in (8, 128, 264, 1000, 1024, 2048, 2176, 4096, 8192, 8200, 8320)
                     for n in (1, 64, 128, 129, 256, 257, 258, 320, 512, 513, 1000) for s in (1, 4)}


def test_every_form_of_a_decode_product_of_the_inputs_is_run():
    from tests.test_gpu_hybrid import FORMS
    lib = _lib.load_dense()
    forms = {lib.ajqd_dense_in_form(batch, k, width // 16, 0) for batch, k, width in FORMS}
    assert forms == {221110, 221210, 821214, 422214, 422210, 421110, 421121, 421112, 421114}
    assert forms | {421210} == {lib.ajqd_dense_in_form(b, k, n, m) for b in (1, 3, 5, 8, 9, 17, 33, 64) for k in (8, 128, 264, 1000, 1024, 2048, 2176, 4096, 8192, 8200)
                                for n in (0, 1, 64, 129, 256, 320, 1000) for m in (0, 2, 128, 400) if n + m}


@pytest.mark.parametrize("batch,k,tiles1,tiles2,form", [  # two blocks of columns at a time, and not in a round that is nearly full or past 384 tiles
    (1, 2048, 192, 0, 421121), (1, 2048, 0, 194, 421110), (4, 4096, 256, 0, 421110), (2, 2048, 129, 128, 421121), (4, 2048, 384, 0, 421121), (4, 2048, 385, 0, 421110),
    (4, 1024, 64, 0, 421110), (4, 2176, 64, 0, 421110), (5, 2048, 64, 0, 421112), (33, 2048, 128, 0, 821214), (33, 2048, 129, 0, 422214),
])
def test_form_of_a_decode_product_of_the_inputs(batch, k, tiles1, tiles2, form):
    assert _lib.load_dense().ajqd_dense_in_form(batch, k, tiles1, tiles2) == form


@pytest.mark.parametrize("batch,k,width,form", [  # few sequences: staged rows on both sides of each line
    (1, 2048, 1024, 811111), (1, 2176, 1024, 811110), (4, 3072, 2048, 811111), (4, 2560, 2048, 811110), (1, 4096, 4096, 421110), (1, 4096, 4112, 421111),
    (1, 4096, 6144, 421111), (1, 4096, 6160, 421110), (4, 8192, 4096, 421121), (4, 9216, 4096, 421110), (4, 9216, 3072, 421121), (1, 8320, 3072, 421111),
    (5, 2176, 4096, 421110), (5, 2560, 4096, 421112), (5, 2176, 4112, 421112), (6, 3200, 4096, 421110), (7, 3200, 4096, 421112), (6, 3584, 4096, 421112), (9, 2176, 4096, 421114),
])
def test_form_of_a_decode_product_of_few_sequences(batch, k, width, form):
    assert _lib.load_dense().ajqd_dense_out_form(batch, k, width, 0, 0) == form


@pytest.mark.parametrize("streams,batch,k,width,scaled,form", [
    # more than four streams and 16 sequences on 16-row tiles: from memory, one tile, one block, up to rows of 8192 columns
    (12, 33, 1152, 2064, 1, 421210), (5, 17, 1024, 8192, 1, 421210), (16, 64, 8064, 4096, 0, 421210),
    (8, 64, 8192, 4096, 1, 422214), (16, 17, 8192, 2064, 1, 421214), (8, 64, 8200, 8192, 1, 421210),
    # and the forms beside it: 8-row tiles, up to four streams, up to 16 sequences
    (12, 64, 1024, 512, 1, 811214), (4, 33, 1152, 2064, 1, 421214), (4, 33, 1152, 4096, 1, 422214), (4, 17, 2056, 4096, 1, 421220), (16, 16, 4096, 4096, 1, 421114),
    # two blocks at a time: rows off the grid that are long for their streams, and up to 16 sequences
    (6, 31, 16024, 2976, 0, 421220), (6, 33, 16024, 2976, 0, 421210), (16, 31, 16024, 2976, 0, 421210), (5, 17, 8184, 2976, 0, 421210), (5, 17, 8200, 2976, 0, 421220),
    (5, 12, 16384, 4096, 0, 421114), (5, 8, 16384, 4096, 1, 421122), (4, 9, 16384, 4096, 1, 421124), (1, 12, 11264, 4096, 0, 421114), (1, 16, 10240, 4096, 0, 421124),
    (1, 16, 9216, 4096, 0, 421114),
])
def test_form_of_a_decode_product_with_streams(streams, batch, k, width, scaled, form):
    assert _lib.load_dense().ajqd_dense_out_form(batch, k, width, streams, scaled) == form


@pytest.mark.parametrize("units,share,dimp,chunks,better", [
    (512, 16, 128, 32, 1), (26, 16, 128, 10, 1), (128, 7, 144, 2, 1), (128, 1, 160, 2, 1), (129, 4, 160, 2, 0), (26, 16, 160, 10, 0), (4, 8, 144, 32, 0), (65, 8, 144, 2, 1),
    (64, 11, 160, 4, 1), (64, 12, 160, 4, 0), (4, 17, 128, 4, 0), (4, 4, 176, 4, 0),
])
def test_one_launch_for_the_decode_attention_where_it_is_the_faster(units, share, dimp, chunks, better):
    assert _lib.load_dense().ajqd_group_decode_better(units, share, dimp, 64, chunks) == better


def test_decode_attention_that_makes_its_row_refuses_bad_arguments():
    lib = _lib.load_dense()
    buf = ctypes.create_string_buffer(4096)
    p = ctypes.c_void_p((ctypes.addressof(buf) + 15) & ~15)
    args = _lib.KeyValueSplitArgs(y=p, q_gain=p, k_gain=p, half_turns=p, pos=p, rows=p, tokens=1, seq=1, ldy=64, heads=2, groups=2, dim=16, dimp=16, rot=8,
                                  cap=4, kept=0, rows_head=128, rows_batch=256)
    run = lambda chunks=1: lib.ajqd_group_decode(ctypes.byref(args), p, chunks, 1.0, None)
    assert run(0) == -2 and run(33) == -2
    for name, value, code in (("pos", None, -1), ("half_turns", None, -1), ("seq", 2, -2), ("heads", 3, -2), ("kept", 4, -2), ("rows_head", 160, -2), ("prior", 1, -2),
                              ("rows_batch", 288, -2), ("ldy", 60, -2), ("rot", 6, -4), ("rot", 18, -2)):
        before = getattr(args, name)
        setattr(args, name, value)
        assert run() == code, name
        setattr(args, name, before)
    args.y = ctypes.c_void_p(p.value + 4)
    assert run() == -3
