"""Prefill-form expert GEMMs at the edges of their K pipelines and token tiles.

Two experts that every token picks, so each holds T positions, T around the
16-position column tiles and the 64-position tiles.  The pipelines' loops take
six stages a round and up to five after it: int4 runs H / 128 stages in gate_up
(H is a multiple of 256, so remainders 0, 2 and 4) and I / 128 in down
(remainders 0 .. 5, with and without a full round before them); int8 and bf16
run H / 64 and I / 64, both even (0, 2, 4).

Small batches are checked against the oracle (tolerance as in
moe_cases.compare, bf16 outputs): int4 there runs eight waves per workgroup,
bf16's gate_up the register-staged kernel from 60 positions on.  Large batches, where
int4 runs four waves and bf16 its pipeline, are checked bit for bit against
the small ones."""
from dataclasses import replace

import pytest
import torch

from moe_cases import CONFIGS, Layer, build_inputs, build_layer, compare, native_layer, oracle_forward

pytestmark = pytest.mark.gpu

# (H, I) in 128-wide stages: 2/1, 4/3, 6/5, 8/2, 10/7, 2/4, 12/6, 2/11, 4/8, 6/9, 2/10
SHAPES = [(256, 128), (512, 384), (768, 640), (1024, 256), (1280, 896), (256, 512), (1536, 768), (256, 1408),
          (512, 1024), (768, 1152), (256, 1280)]


@pytest.mark.parametrize("wfmt", ["int4_g128", "bf16", "int8_per_channel"])
@pytest.mark.parametrize("H,I", SHAPES)
def test_stage_and_tile_remainders(gpu_device, wfmt, H, I):
    cfg = replace(CONFIGS["qwen3_int4"], name=f"stages_{wfmt}", H=H, I=I, E=2, k=2, wfmt=wfmt)
    layer = build_layer(cfg, device="cuda")
    native = native_layer(layer, torch.device("cuda"))
    # last tiles of 13 .. 64 positions alone, of 1, 2, 16, 26, 41 and 56 after a full one
    for T in (13, 17, 33, 49, 64, 65, 130, 80, 90, 105, 120):
        x, logits = build_inputs(layer, T, seed=T, device="cuda")
        out = native.forward(x, logits)
        torch.cuda.synchronize()
        ref = oracle_forward(layer, x, logits)
        compare(out.float().cpu().numpy(), ref, cfg)


@pytest.mark.parametrize("wfmt", ["int4_g128", "bf16", "int8_per_channel"])
@pytest.mark.parametrize("H,I", SHAPES)
def test_stage_and_tile_remainders_in_large_batches(gpu_device, wfmt, H, I):
    """Batches of more than 272 (tile, slab) items in either projection and
    more than 256 positions per expert whose last tile holds r: its rows, and
    the first full tile's, have the bits of a batch of those tokens alone."""
    cfg = replace(CONFIGS["qwen3_int4"], name=f"stages_{wfmt}", H=H, I=I, E=2, k=2, wfmt=wfmt)
    layer = build_layer(cfg, device="cuda")
    native = native_layer(layer, torch.device("cuda"), max_tokens=9000)
    slabs = min(I // 128, H // 256)
    full = max(5, (272 // slabs) // 2 + 1)  # full tiles of each expert: slabs * (2 full + 1) > 272
    x, logits = build_inputs(layer, 64 * full + 64, seed=7, device="cuda")
    first = native.forward(x[:64].contiguous(), logits[:64].contiguous()).clone()
    for r in (13, 26, 41, 57, 64):
        T = 64 * full + r
        out = native.forward(x[:T].contiguous(), logits[:T].contiguous()).clone()
        alone = native.forward(x[64 * full:T].contiguous(), logits[64 * full:T].contiguous())
        torch.cuda.synchronize()
        assert torch.equal(out[64 * full:], alone), f"last tile of {r}"
        assert torch.equal(out[:64], first), f"first tile, r = {r}"


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


@pytest.mark.parametrize("wfmt", ["int4_g128", "bf16", "int8_per_channel"])
def test_rows_at_any_address(gpu_device, wfmt):
    """hidden_states that start between 16-byte boundaries (a contiguous view
    one element into its storage) give the bits of an aligned copy, in the
    decode form (T = 3) and the prefill form."""
    cfg = replace(CONFIGS["qwen3_int4"], name=f"offset_{wfmt}", H=512, I=384, E=2, k=2, wfmt=wfmt)
    layer = build_layer(cfg, device="cuda")
    native = native_layer(layer, torch.device("cuda"))
    for T in (3, 33, 130):
        x, logits = build_inputs(layer, T, seed=T, device="cuda")
        store = torch.zeros(x.numel() + 16, dtype=x.dtype, device="cuda")
        view = store[1:1 + x.numel()].view(T, cfg.H)
        view.copy_(x)
        assert view.data_ptr() % 16 == 2
        aligned = native.forward(x, logits).clone()
        offset = native.forward(view, logits)
        torch.cuda.synchronize()
        assert torch.equal(aligned, offset), f"T = {T}"
