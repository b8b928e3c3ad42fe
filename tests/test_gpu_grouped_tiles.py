"""The list of tiles that the grouped W4A16 GEMMs go over: every expert has exactly T pairs, T on both sides of a 32-token block
and of a tile's 128 tokens, through the prefill layer (the list is made from 5 tokens on) and through the decode layer with its
matrix-core classes (flags 0x600, where the list is made from 129 tokens on).  Oracle: the layer in the reference's schedule
(src/kimi_exec.cu:835-877); bound: 1e-2 of the largest element, which the bf16 roundings of a layer stay below (0.5e-2 measured with
other orders of the sums)."""
import ctypes as C

import numpy as np
import pytest

import oracle as O
from blok_amd.lib import check
from kxt import dev, moe_case, moe_cfg, moe_device_weights, moe_oracle_weights

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("path,T", [("prefill", t) for t in (1, 4, 5, 31, 97, 128, 129, 257)] + [("decode", t) for t in (6, 128, 129, 161)])
def test_every_expert_has_all_tokens(kxlib, ox, path, T):
    H, I, SI, E, K = 1024, 1024, 512, 3, 3
    print(f"grouped tiles {path} T={T}", flush=True)
    host, n, x = moe_case(kxlib, H, I, SI, E, K, T, 77)
    cfg = moe_cfg(H, I, SI, E, K)
    w, bufs = moe_device_weights(host)
    ws = C.c_void_p()
    check(kxlib.kx_moe_workspace_create(C.byref(cfg), T, C.byref(ws)))
    dn, dx = dev(n), dev(x)
    call, flags = (kxlib.kx_moe_prefill_layer, 0) if path == "prefill" else (kxlib.kx_moe_decode_layer, 0x600)
    check(call(C.byref(cfg), C.byref(w), ws, dn.ptr, dx.ptr, T, flags, None))
    check(kxlib.kx_sync(None))
    got = dx.to_numpy(np.uint16, (T, H))
    check(kxlib.kx_moe_workspace_destroy(ws))
    want, wo = x.copy(), moe_oracle_weights(host)
    ox.ox_moe_layer(C.byref(wo), n.ctypes.data, want.ctypes.data, T, H, I, SI, E, K, 2.827, 0, 0, None, None, None, None, None)
    err = O.max_rel(O.bf16_to_f32(got), O.bf16_to_f32(want))
    assert err < 1e-2, err


def _run(kxlib, host, n, x, H, I, SI, E, K, T, path, flags):
    """The layer, with expert outputs that show where nothing is written."""
    cfg = moe_cfg(H, I, SI, E, K)
    w, bufs = moe_device_weights(host)
    ws = C.c_void_p()
    check(kxlib.kx_moe_workspace_create(C.byref(cfg), T, C.byref(ws)))
    views = [C.c_void_p() for _ in range(8)]
    check(kxlib.kx_moe_workspace_views(ws, *(C.byref(v) for v in views)))
    for v, width in ((views[6], I), (views[7], H)):
        check(kxlib.kx_dev_memset(v, 0x7f, T * K * width * 2, None))
    dn, dx = dev(n), dev(x)
    call = kxlib.kx_moe_prefill_layer if path == "prefill" else kxlib.kx_moe_decode_layer
    check(call(C.byref(cfg), C.byref(w), ws, dn.ptr, dx.ptr, T, flags, None))
    check(kxlib.kx_sync(None))
    got = dx.to_numpy(np.uint16, (T, H))
    check(kxlib.kx_moe_workspace_destroy(ws))
    return got


@pytest.mark.parametrize("path,T,E", [("decode", t, 8) for t in (9, 31, 32, 40, 64, 65, 128, 129)] + [("prefill", 31, 8)] +
                         [("plain", t, e) for t, e in ((1, 8), (4, 8), (9, 80), (10, 80), (32, 8), (64, 8))])
def test_fewer_candidates_than_choices(kxlib, ox, path, T, E):
    """All experts but three have a bias of -inf: expert 0 stands for the missing choices of every token as well (src/kimi_exec.cu:391-393)
    and has six pairs per token, more than a tile holds and more than there are tokens."""
    H, I, SI, K = 1024, 1024, 512, 8
    print(f"masked experts {path} T={T} E={E}", flush=True)
    host, n, x = moe_case(kxlib, H, I, SI, E, K, T, 78)
    host = dict(host, router_bias=host["router_bias"].copy())
    host["router_bias"][[e for e in range(E) if e not in (0, 3, 5)]] = -np.inf
    got = _run(kxlib, host, n, x, H, I, SI, E, K, T, path, 0x600 if path == "decode" else 0)
    want, wo = x.copy(), moe_oracle_weights(host)
    ox.ox_moe_layer(C.byref(wo), n.ctypes.data, want.ctypes.data, T, H, I, SI, E, K, 2.827, 0, 0, None, None, None, None, None)
    err = O.max_rel(O.bf16_to_f32(got), O.bf16_to_f32(want))
    assert err < 1e-2, err


@pytest.mark.parametrize("path,T", [("decode", 129), ("decode", 161), ("decode", 300), ("prefill", 161)])
def test_experts_of_every_class_beside_each_other(kxlib, ox, path, T):
    """Experts with all tokens, with 1, 2, 3, 33 and 97 of them and with none: those of 1 and 2 pairs are no tiles of the decode layer,
    another kernel computes them at the same time.  What no kernel writes shows."""
    H, I, SI, E, K = 1024, 1024, 512, 12, 3
    print(f"classes {path} T={T}", flush=True)
    host, n, x = moe_case(kxlib, H, I, SI, E, K, T, 79)
    order = np.random.default_rng(T).permutation(E)                                 # so that the classes are not in the order of their sizes
    pick, at = np.zeros((T, E), bool), 0
    pick[:, order[0]] = True
    for e, count in zip(order[1:], (1, 2, 3, 33, 97)):
        pick[(at + np.arange(count)) % T, e] = True
        at += count
    for t in range(T):                                                              # the rest to two experts
        pick[t, order[6:8][:K - pick[t].sum()]] = True
    assert (pick.sum(1) == K).all() and pick.sum(0)[order[:6]].tolist() == [T, 1, 2, 3, 33, 97] and (pick.sum(0) == 0).sum() >= 4
    host = dict(host, router_gate=np.zeros((E, H), np.float32), router_bias=np.zeros(E, np.float32))
    host["router_gate"][np.arange(E), np.arange(E)] = 4.0
    host["router_gate"] = (host["router_gate"].view(np.uint32) >> 16).astype(np.uint16).reshape(-1)
    n = n.copy()
    n[:, :E] = (np.where(pick, 2.0, -2.0).astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)
    got = _run(kxlib, host, n, x, H, I, SI, E, K, T, *(("prefill", 0) if path == "prefill" else ("decode", 0x600)))
    want, wo = x.copy(), moe_oracle_weights(host)
    ox.ox_moe_layer(C.byref(wo), n.ctypes.data, want.ctypes.data, T, H, I, SI, E, K, 2.827, 0, 0, None, None, None, None, None)
    err = O.max_rel(O.bf16_to_f32(got), O.bf16_to_f32(want))
    assert err < 1e-2, err


def test_scratch_of_a_small_workspace(kxlib):
    """The parts of its products' columns: 16 MiB for the router and as much for the shared expert, where the tiles are few."""
    cfg = moe_cfg(1024, 1024, 512, 32, 4)
    free, total = [], C.c_size_t()
    for make in (False, True):
        ws = C.c_void_p()
        if make:
            check(kxlib.kx_moe_workspace_create(C.byref(cfg), 64, C.byref(ws)))
        free.append(C.c_size_t())
        check(kxlib.kx_dev_mem_info(C.byref(free[-1]), C.byref(total)))
        if make:
            check(kxlib.kx_moe_workspace_destroy(ws))
    assert free[0].value - free[1].value < 64 << 20, (free[0].value - free[1].value) >> 20
