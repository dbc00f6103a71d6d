"""GPU Qwen3 encodes of few token rows (at most 128 in bf16, 64 in f32), which
run on kernels of their own, against the numpy oracle (oracle/qwen3.py).

Two layers of random weights at shapes that cover both hidden widths the path
takes, one, two and four query heads per K/V head, and row counts at the edges
of its 16-row blocks, of its text-length classes (32, 64, 128) and of the path
itself. Tolerances are those of the general path's own test
(tests/test_qwen3_e2e_gpu.py): f32 cosine 0.99999 and 2e-4 max-abs, bf16
cosine 0.999 on the bf16-rounded weights; and, a text at a time, relative
distances at twice what right code shows. f32 4e-6. bf16 1.6e-2, of roundings to
8 bits in some 20 places of two layers: in the oracle, hiding one key of a text
of 65 to 128 from the rows after it moves its embedding by 6e-2 or more."""
import numpy as np
import pytest

from oracle import attention as oa
from oracle import qwen3 as oq

pytestmark = pytest.mark.gpu

SHAPES = {
    "0.6B": dict(),
    "group1": dict(hidden=512, intermediate=2048, heads=8, kv_heads=8),
    "group4": dict(intermediate=1024, heads=16, kv_heads=4),
}
CASES = [("0.6B", [1]), ("0.6B", [16]), ("0.6B", [17]), ("0.6B", [31, 1]), ("0.6B", [33]), ("0.6B", [5, 1, 32, 10]),
         ("0.6B", [64]), ("0.6B", [65]), ("0.6B", [127]), ("0.6B", [3, 97, 28]), ("0.6B", [100, 29]),
         ("group1", [23]), ("group1", [40, 24]), ("group4", [23]), ("group4", [64]), ("group4", [80])]


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("shape,lengths", CASES)
def test_few_rows_against_oracle(shape, lengths, dtype, cuda, inl):
    import torch
    cfg = oq.Qwen3Config(vocab=512, layers=2, **SHAPES[shape])
    w = oq.random_weights(cfg, seed=11)
    td = torch.float32 if dtype == "f32" else torch.bfloat16
    wd = {k: torch.from_numpy(np.ascontiguousarray(v)).to(cuda).to(td) for k, v in w.items()}
    if dtype == "bf16":
        w = {k: v.float().cpu().numpy() for k, v in wd.items()}
    rng = np.random.default_rng(sum(lengths))
    cu = oa.cu_from_lengths(lengths)
    enc = inl.Qwen3Encoder(cfg, wd, max_positions=128)
    print(f"case={shape} {dtype} {lengths}", flush=True)
    for call in range(3):   # eager, captured and replayed
        ids = rng.integers(0, cfg.vocab, sum(lengths))
        got = enc.encode(ids, cu.tolist()).cpu().numpy().astype(np.float64)
        ref = oq.encode(w, cfg, ids, cu)
        cos = (got * ref).sum(1) / np.linalg.norm(got, axis=1) / np.linalg.norm(ref, axis=1)
        rel = (np.linalg.norm(got - ref, axis=1) / np.linalg.norm(ref, axis=1)).max()
        print(f"relative error {rel:.3g}", flush=True)
        if dtype == "f32":
            assert cos.min() >= 0.99999 and np.abs(got - ref).max() <= 2e-4 and rel <= 4e-6
        else:
            assert cos.min() >= 0.999 and rel <= 1.6e-2
    enc.close()


# A caller may size one workspace for its largest batch: a smaller batch needs
# no more of it, also where it moves to the few-row kernels.
@pytest.mark.parametrize("dtype,rows", [("f32", 64), ("bf16", 128)])
def test_few_rows_need_no_larger_workspace(dtype, rows, cuda, inl):
    import torch
    cfg = oq.Qwen3Config(vocab=512, layers=1)
    td = torch.float32 if dtype == "f32" else torch.bfloat16
    wd = {k: torch.from_numpy(np.ascontiguousarray(v)).to(cuda).to(td) for k, v in oq.random_weights(cfg, seed=13).items()}
    enc = inl.Qwen3Encoder(cfg, wd, max_positions=512)
    sizes = [enc.workspace_bytes([0, n]) for n in (1, rows - 1, rows, rows + 1)]
    enc.close()
    assert sizes == sorted(sizes)


# f32 batches above 464 rows run on the library's own f32 GEMM: row counts at
# the edges of its 128-row tiles and of the path, and widths with other part
# counts. The tolerance of the general path, and a relative distance of 2.5e-6
# (two layers of f32 sums: 4e-7 to 6e-7, on hipBLASLt 1.3e-6): weights cut to two
# of their three bf16 parts move the oracle by 8e-6. (The group1 batch of 513 rows
# has too few tiles and runs on hipBLASLt.)
@pytest.mark.parametrize("shape,lengths", [("0.6B", [465]), ("0.6B", [200, 312]), ("0.6B", [300, 200, 140, 1]),
                                           ("group1", [500, 13]), ("group4", [512, 257]), ("group1", [500, 200])])
def test_f32_gemm_rows_against_oracle(shape, lengths, cuda, inl):
    import torch
    cfg = oq.Qwen3Config(vocab=512, layers=2, **SHAPES[shape])
    w = oq.random_weights(cfg, seed=12)
    wd = {k: torch.from_numpy(np.ascontiguousarray(v)).to(cuda) for k, v in w.items()}
    rng = np.random.default_rng(sum(lengths))
    cu = oa.cu_from_lengths(lengths)
    ids = rng.integers(0, cfg.vocab, sum(lengths))
    print(f"case=f32_gemm {shape} {lengths}", flush=True)
    enc = inl.Qwen3Encoder(cfg, wd, max_positions=512)
    got = enc.encode(ids, cu.tolist()).cpu().numpy().astype(np.float64)
    enc.close()
    ref = oq.encode(w, cfg, ids, cu)
    cos = (got * ref).sum(1) / np.linalg.norm(got, axis=1) / np.linalg.norm(ref, axis=1)
    assert cos.min() >= 0.99999 and np.abs(got - ref).max() <= 2e-4
    rel = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    print(f"relative error {rel:.3g}", flush=True)
    assert rel <= 2.5e-6


# Weights that are slices of a larger buffer, one element off a 16-byte boundary:
# the few-row and f32-GEMM kernels load 16 bytes at a time, so such a model takes
# the general sequence, for which unaligned row norms are ordinary and unaligned
# q/k norms an error. Against the encode of the same weights, aligned, within the
# sum of both paths' distances from the oracle above.
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("rows", [17, 500])
def test_unaligned_weights(rows, dtype, cuda, inl):
    import torch
    cfg = oq.Qwen3Config(vocab=512, layers=1)
    td = torch.float32 if dtype == "f32" else torch.bfloat16
    wd = {k: torch.from_numpy(np.ascontiguousarray(v)).to(cuda).to(td) for k, v in oq.random_weights(cfg, seed=14).items()}
    ids = np.random.default_rng(rows).integers(0, cfg.vocab, rows)

    def shifted(name):
        buf = torch.empty(wd[name].numel() + 1, dtype=td, device=cuda)
        buf[1:] = wd[name].reshape(-1)
        view = buf[1:].view(wd[name].shape)
        assert view.data_ptr() % 16 == view.element_size()
        return {**wd, name: view}

    def encode(weights):
        enc = inl.Qwen3Encoder(cfg, weights, max_positions=512)
        try:
            return enc.encode(ids, [0, rows]).cpu().numpy()
        finally:
            enc.close()

    print(f"case=unaligned weights {dtype} rows={rows}", flush=True)
    want = encode(wd)
    for name in ("input_layernorm.weight", "post_attention_layernorm.weight"):
        got = encode(shifted("layers.0." + name))
        cos = (got * want).sum(1) / np.linalg.norm(got, axis=1) / np.linalg.norm(want, axis=1)
        assert cos.min() >= (1 - 2e-5 if dtype == "f32" else 1 - 2e-3)
    for name in ("q_norm.weight", "k_norm.weight"):
        with pytest.raises(inl.InlError):
            encode(shifted("layers.0.self_attn." + name))


# A gate row of the lowest f32 value: its products are finite (silu gives -0),
# but it has no bf16 parts. Within the f32 tolerance of the oracle.
def test_f32_gemm_lowest_weight(cuda, inl):
    import torch
    cfg = oq.Qwen3Config(vocab=64, layers=1, hidden=512, intermediate=256, heads=8, kv_heads=8)
    w = oq.random_weights(cfg, seed=15)
    w["embed_tokens.weight"][:, 0] = np.abs(w["embed_tokens.weight"][:, 0]) + 0.01   # x[0] > 0 at the gate
    w["layers.0.self_attn.o_proj.weight"][0] = 0
    w["layers.0.post_attention_layernorm.weight"][0] = 0.01
    gate = w["layers.0.mlp.gate_proj.weight"]
    gate[[3, 130]] = 0
    gate[[3, 130], 0] = np.finfo(np.float32).min
    wd = {k: torch.from_numpy(np.ascontiguousarray(v)).to(cuda) for k, v in w.items()}
    ids = np.random.default_rng(1).integers(0, cfg.vocab, 700)
    cu = [0, 300, 700]
    print("case=f32_gemm lowest weight", flush=True)
    enc = inl.Qwen3Encoder(cfg, wd, max_positions=512)
    got = enc.encode(ids, cu).cpu().numpy().astype(np.float64)
    enc.close()
    with np.errstate(over="ignore"):
        ref = oq.encode(w, cfg, ids, cu)
    assert np.isfinite(ref).all() and np.abs(got - ref).max() <= 1e-6
