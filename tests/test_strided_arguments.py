"""Non-contiguous inputs of the entry points that copy them: every copy lives until the library has its address. (A copy
freed while the call's arguments are collected hands its memory to the next copy of the same size.)"""
import ctypes
import importlib

import pytest
import torch

LIB = importlib.import_module("b70-inference_amd._lib")
LINEAR = importlib.import_module("b70-inference_amd.linear")
MOE = importlib.import_module("b70-inference_amd.moe")


def columns(g, n, count, dtype):
    """`count` columns of one [n, count] table, and their values."""
    if dtype == torch.float16:
        t = torch.randint(0, 2, (n, count), generator=g).to(dtype) * 2 - 1
    else:
        t = torch.randint(0, 1 << 30, (n, count), generator=g).to(dtype)
    return [t[:, i] for i in range(count)]


def record(monkeypatch, name, sizes):
    """Calls of library function `name` copy what the pointer arguments `sizes` (position -> bytes) lead to."""
    got = {}

    def call(*args):
        for i, n in sizes.items():
            got[i] = ctypes.string_at(args[i], n)
        return 0

    fake = type("Fake", (), {name: staticmethod(call)})()
    for m in (LINEAR, MOE):
        monkeypatch.setattr(m, "lib", lambda: fake)
        monkeypatch.setattr(m, "require_device", lambda *t: None)
        monkeypatch.setattr(m, "stream_of", lambda t: None)
    return got


def raw(t):
    return t.contiguous().numpy().tobytes()


@pytest.mark.parametrize("entry", ["gemm", "gemm_noalloc", "reconstruct_had_slice", "mgemm", "moe_align"])
def test_addresses_are_those_of_each_argument(monkeypatch, entry):
    g = torch.Generator().manual_seed(3)
    k = n = 256
    A, C = torch.zeros(4, k, dtype=torch.float16), torch.zeros(4, n, dtype=torch.float32)
    B = torch.zeros(k // 16, n // 16, 48, dtype=torch.int16)
    suh, svh = columns(g, k, 2, torch.float16)
    if entry in ("gemm", "gemm_noalloc"):
        at = (10, 12) if entry == "gemm" else (10, 11)
        got = record(monkeypatch, "exl3_" + entry, {at[0]: 2 * k, at[1]: 2 * n})
        LINEAR.exl3_gemm(A, B, C, suh, None, svh) if entry == "gemm" else LINEAR.exl3_gemm_noalloc(A, B, C, suh, svh)
        want = {at[0]: raw(suh), at[1]: raw(svh)}
    elif entry == "reconstruct_had_slice":
        got = record(monkeypatch, "exl3_reconstruct_had_slice", {5: 2 * k, 6: 2 * n})
        LINEAR.reconstruct_had_slice(torch.zeros(k, n, dtype=torch.float16), B, suh, svh, 3, False, True, 0)
        want = {5: raw(suh), 6: raw(svh)}
    elif entry == "mgemm":
        tab = columns(g, 64, 3, torch.int64)
        got = record(monkeypatch, "exl3_mgemm", {4: 512, 5: 512, 6: 512})
        LINEAR.exl3_mgemm(A, tab[0], torch.zeros(64, 4, n), tab[1], None, tab[2], None, None, 3)
        want = {4 + i: raw(t) for i, t in enumerate(tab)}
    else:
        ids = torch.randint(0, 8, (96, 8), generator=g, dtype=torch.int32)[:, ::2]
        w = torch.rand(96, 8, generator=g)[:, ::2]
        got = record(monkeypatch, "exl3_moe_align", {0: 4 * ids.numel(), 1: 4 * w.numel()})
        MOE.moe_align(ids, w, 8)
        want = {0: raw(ids), 1: raw(w)}
    assert got == want


@pytest.mark.gpu
@pytest.mark.parametrize("entry", ["gemm", "gemm_noalloc", "reconstruct_had_slice", "mgemm", "moe_align"])
def test_strided_inputs_give_the_contiguous_results(exl3, entry):
    g = torch.Generator().manual_seed(4)
    k = n = 256
    dev = "cuda"
    A = torch.randn(4, k, generator=g).half().to(dev)
    B = [torch.randint(-32768, 32768, (k // 16, n // 16, 48), generator=g, dtype=torch.int16).to(dev) for _ in range(3)]
    signs = torch.stack(columns(g, k, 2, torch.float16), 1).to(dev)
    suh, svh = signs[:, 0], signs[:, 1]

    def run(suh, svh, strided):
        if entry == "gemm":
            C = torch.empty(4, n, device=dev)
            exl3.exl3_gemm(A, B[0], C, suh, None, svh)
            return [C]
        if entry == "gemm_noalloc":
            C = torch.empty(4, n, device=dev)
            exl3.exl3_gemm_noalloc(A, B[0], C, suh, svh)
            return [C]
        if entry == "reconstruct_had_slice":
            W = torch.empty(k, n, dtype=torch.float16, device=dev)
            exl3.reconstruct_had_slice(W, B[0], suh, svh, 3, False, True, 0)
            return [W]
        if entry == "mgemm":
            s = [t.contiguous() for t in (signs[:, 0], signs[:, 1])]
            tab = torch.tensor([[b.data_ptr(), s[0].data_ptr(), s[1].data_ptr()] for b in B], device=dev)
            cols = [tab[:, i] if strided else tab[:, i].contiguous() for i in range(3)]
            C = torch.empty(3, 4, n, device=dev)
            exl3.exl3_mgemm(A, cols[0], C, cols[1], None, cols[2], None, None, 3)
            torch.cuda.synchronize()
            return [C]
        ids, w = torch.stack([torch.randperm(8, generator=torch.Generator().manual_seed(i)) for i in range(40)]).int(), \
            torch.rand(40, 8, generator=torch.Generator().manual_seed(9))
        ids, w = ids.to(dev)[:, ::2], w.to(dev)[:, ::2]
        if not strided:
            ids, w = ids.contiguous(), w.contiguous()
        counts, tok, wt, _ = exl3.moe_align(ids, w, 8)
        e = torch.repeat_interleave(torch.arange(8, device=dev), counts.long())
        order = torch.argsort(e * 64 + tok)                     # (the order within an expert is free)
        return [counts, tok[order], wt[order]]

    for a, b in zip(run(suh, svh, True), run(suh.contiguous(), svh.contiguous(), False)):
        assert torch.equal(a, b)
