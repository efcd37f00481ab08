"""Prefill-form expert GEMMs at the edges of their K pipelines and token tiles.

Two experts that every token picks, so each holds T positions: T around the
16-position column tiles and the 64-position tiles, and H / I so that gate_up
and down end in every remainder of the unrolled stage loop (1 .. 8 stages of
128).  Tolerance as in moe_cases.compare (bf16 outputs)."""
from dataclasses import replace

import pytest
import torch

from moe_cases import CONFIGS, Layer, build_inputs, build_layer, compare, native_layer, oracle_forward

pytestmark = pytest.mark.gpu

# (H, I): gate_up runs H / 128 stages, down I / 128
SHAPES = [(256, 128), (512, 384), (768, 640), (1024, 256), (1280, 896), (256, 512)]


@pytest.mark.parametrize("wfmt", ["int4_g128", "bf16", "int8_per_channel"])
@pytest.mark.parametrize("H,I", SHAPES)
def test_stage_and_tile_remainders(gpu_device, wfmt, H, I):
    cfg = replace(CONFIGS["qwen3_int4"], name=f"stages_{wfmt}", H=H, I=I, E=2, k=2, wfmt=wfmt)
    layer = build_layer(cfg, device="cuda")
    native = native_layer(layer, torch.device("cuda"))
    for T in (13, 17, 33, 49, 64, 65, 130):
        x, logits = build_inputs(layer, T, seed=T, device="cuda")
        out = native.forward(x, logits)
        torch.cuda.synchronize()
        ref = oracle_forward(layer, x, logits)
        compare(out.float().cpu().numpy(), ref, cfg)


def test_int4_rows_same_bits_in_every_batch(gpu_device):
    """An int4 prefill row does not depend on the batch it is in: few experts
    at token counts on both sides of one (tile, slab) item per CU, where
    gate_up (16 slabs) and then down (8 slabs) go from eight waves per
    workgroup to four -- both on eight up to T = 256 (at most 192 items),
    gate_up on four at 400, both at 1024 -- give bit-identical prefixes."""
    cfg = replace(CONFIGS["qwen3_int4"], name="few_experts_int4", H=2048, I=2048, E=8, k=2)
    layer = build_layer(cfg, device="cuda")
    native = native_layer(layer, torch.device("cuda"))
    x, logits = build_inputs(layer, 1024, seed=3, device="cuda")
    full = native.forward(x, logits).clone()
    compare(full[:97].float().cpu().numpy(), oracle_forward(layer, x[:97], logits[:97]), cfg)
    for T in (33, 64, 180, 256, 400, 900):
        assert not cfg.decode_form(T)
        part = native.forward(x[:T].contiguous(), logits[:T].contiguous())
        torch.cuda.synchronize()
        assert torch.equal(full[:T], part), f"T = {T}"


def test_bf16_rows_same_bits_in_every_batch(gpu_device):
    """A bf16 prefill row does not depend on the batch either: experts of 20
    MiB whose gate_up leaves the stage pipeline for the register-staged form
    from 60 to 255 positions per expert (T = 300, 1000), and whose down (K =
    4096, 5 slabs) leaves it up to 273 (tile, slab) items (T = 2200 above)."""
    cfg = replace(CONFIGS["qwen3_int4"], name="few_experts_bf16", H=1280, I=4096, E=8, k=2, wfmt="bf16")
    layer = build_layer(cfg, device="cuda")
    native = native_layer(layer, torch.device("cuda"))
    x, logits = build_inputs(layer, 2200, seed=5, device="cuda")
    full = native.forward(x, logits).clone()
    compare(full[:97].float().cpu().numpy(), oracle_forward(layer, x[:97], logits[:97]), cfg)
    for T in (97, 300, 1000, 1500):
        assert not cfg.decode_form(T)
        part = native.forward(x[:T].contiguous(), logits[:T].contiguous())
        torch.cuda.synchronize()
        assert torch.equal(full[:T], part), f"T = {T}"


def test_bf16_expert_past_2_gib(gpu_device):
    """One expert whose gate_up takes 2 GiB (the up rows past 1 GiB, the last
    ones close to 2): gemm2_kernel's range, against the same products in
    fp32 on the same bf16 values.  Tolerance as in moe_cases.compare."""
    H, I, T = 4096, 131072, 70
    cfg = replace(CONFIGS["qwen3_int4"], name="bf16_2gib", H=H, I=I, E=1, k=1, wfmt="bf16")
    g = torch.Generator(device="cuda").manual_seed(9)

    def randn(n, k, std):
        return torch.empty(n, k, dtype=torch.bfloat16, device="cuda").normal_(0, std, generator=g)

    native = native_layer(Layer(cfg, torch.zeros(1, H), []), torch.device("cuda"), max_tokens=T)
    gate, up, down = randn(I, H, 0.02), randn(I, H, 0.02), randn(H, I, 0.002)  # y of std about 0.6
    native.load_expert(0, gate, up, down)
    x = torch.randn(T, H, device="cuda", generator=g).to(torch.bfloat16)
    out = native.forward(x, torch.zeros(T, 1, dtype=torch.bfloat16, device="cuda"))
    torch.cuda.synchronize()
    ref = torch.zeros(T, H, device="cuda")
    for i in range(0, I, 16384):
        a, b = x.float() @ gate[i:i + 16384].float().T, x.float() @ up[i:i + 16384].float().T
        ref += (torch.nn.functional.silu(a) * b) @ down[:, i:i + 16384].float().T
    compare(out.float().cpu().numpy(), ref.cpu().numpy(), cfg)
