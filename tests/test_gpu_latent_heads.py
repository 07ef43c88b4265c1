"""The heads' own keys and values from a cached latent, and attention on them, against the same computation in float64."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def reference(q, latents, cut, w_k, w_v, table, scale, sink, gate, per_head, R, dr):
    """Keys, values and turned queries rounded to bfloat16 where the kernels round them; everything else float64."""
    H = w_k.shape[0]
    rounded = lambda t: t.float().bfloat16().double()
    q = q.double().view(q.shape[0], H, 128 + dr)
    outs, row = [], 0
    for (count, start), lat in zip(cut, latents):
        c, kr = lat[:, :R].double(), lat[:, R:].double()
        k, v = rounded(torch.einsum("hdr,nr->hnd", w_k.double(), c)), rounded(torch.einsum("hdr,nr->hnd", w_v.double(), c))
        for i in range(count):
            pos, x = start + i, q[row]
            s = torch.einsum("hd,hnd->hn", x[:, :128], k[:, :pos + 1])
            if dr:
                cos, sin = table[pos, :32].double(), table[pos, 32:].double()
                a, b = x[:, 128:160], x[:, 160:]
                s = s + rounded(torch.cat([a * cos - b * sin, b * cos + a * sin], -1)) @ kr[:pos + 1].T
            s = s * scale
            if sink is not None:
                s = torch.cat([s, sink.double()[:, None]], 1)
            w = torch.softmax(s, -1)[:, :pos + 1]
            o = torch.einsum("hn,hnd->hd", w, v[:, :pos + 1])
            if gate is not None:
                g = torch.sigmoid(gate[row].double())
                o = o * (g[:H, None] if per_head else g.view(H, 128))
            outs.append(o.flatten())
            row += 1
    return torch.stack(outs)


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("R, dr, H, ps, cut, gate, sinks", [
    # one to three blocks, ends inside blocks and units; a request behind a context beside whole prompts; walks of several turns
    (256, 64, 2, 16, [(1, 0), (31, 0), (32, 0), (33, 0), (64, 0), (65, 0)], "channel", False),
    (256, 64, 3, 8, [(200, 0), (5, 130), (129, 31)], "head", False),
    (256, 0, 1, 16, [(1, 95), (2, 300), (128, 1)], None, True),
    (128, 64, 2, 32, [(70, 0), (1, 0), (161, 64)], None, False),
    (128, 0, 5, 16, [(97, 0)] + [(2, 3)] * 70, "head", True),
])
def test_against_float64(R, dr, H, ps, cut, gate, sinks, wide, monkeypatch):
    from minivllm_amd.engine.step import AttentionPlan
    from minivllm_amd.kernels.ops import Ops, latent_operands
    from minivllm_amd.parts import Workspace
    ops = Ops(torch.bfloat16)
    monkeypatch.setattr(ops, "compute_units", 0 if wide else 1 << 20)
    gen = torch.Generator().manual_seed(5)
    rand = lambda *shape: torch.randn(*shape, generator=gen)
    lens, starts = [c for c, _ in cut], [s for _, s in cut]
    context = [c + s for c, s in cut]
    n, pad = sum(lens), 3                                  # three rows of no request at the end
    latents = [rand(c, R + dr).bfloat16() for c in context]
    per = [-(-c // ps) for c in context]
    order, at = torch.randperm(sum(per) + 2, generator=gen).tolist(), 0
    pages = torch.full((sum(per) + 2, ps, R + dr), float("nan"))       # slots that were never written
    table_of = torch.full((len(cut) + 1, max(per) + 1), -1, dtype=torch.int32)
    for i, (lat, p) in enumerate(zip(latents, per)):
        table_of[i, :p] = torch.tensor(order[at:at + p], dtype=torch.int32)
        for j in range(p):
            rows = lat[j * ps:(j + 1) * ps]
            pages[order[at + j], :rows.shape[0]] = rows.float()
        at += p
    i32 = lambda x: torch.tensor(list(x), dtype=torch.int32, device=DEV)
    cu = i32([0] + torch.tensor(lens).cumsum(0).tolist() + [n])        # (one request without a token)
    positions = i32([p for c, s in cut for p in range(s, s + c)] + [0] * pad)
    token_seq = i32([i for i, c in enumerate(lens) for _ in range(c)] + [-1] * pad)
    q = (rand(n + pad, H * (128 + dr)) / math.sqrt(128 + dr) * 4).bfloat16()
    w_k, w_v = (rand(H, 128, R) / math.sqrt(R)).bfloat16(), (rand(H, 128, R) / math.sqrt(R)).bfloat16()
    angle = rand(max(context), 32)
    table = torch.cat([angle.cos(), angle.sin()], 1) if dr else None
    sink = rand(H) if sinks else None
    g = rand(n + pad, H if gate == "head" else H * 128).bfloat16() if gate else None
    dev = lambda t: None if t is None else t.to(DEV)
    plan = AttentionPlan(decode_only=False, max_q_len=max(lens), max_context_len=max(context), n_seqs=len(cut) + 1, q_lens=lens + [0],
                         cu_seqlens=cu, workspace=Workspace(torch.device(DEV)), starts=starts)
    blocks = sum(-(-c // 32) for c in context) + 3         # (more than there are)
    k = torch.full((blocks, H, 4096), float("nan"), dtype=torch.bfloat16, device=DEV)
    v, kr = torch.full_like(k, float("nan")), torch.full((blocks, 32 * max(dr, 1)), float("nan"), dtype=torch.bfloat16, device=DEV)
    out = torch.full((n + pad, H * 128), float("nan"), dtype=torch.bfloat16, device=DEV)
    lens_d = i32(context + [0])
    ops.latent_expand(dev(pages).bfloat16(), dev(table_of), ps, plan, lens_d, dev(latent_operands(w_k)), dev(latent_operands(w_v)), H, R, dr, blocks, k, kr, v)
    ops.attention_latent_heads(dev(q), out, k, kr, v, plan, positions, token_seq, lens_d, H, dr, 0.3, dev(table), dev(sink), dev(g), gate == "head")
    want = reference(q[:n], latents, cut, w_k, w_v, table, 0.3, sink, None if g is None else g[:n], gate == "head", R, dr)
    got = out.double().cpu()
    assert not got[n:].abs().max()
    # a weight and the result are rounded to eight bits each, 2^-9 of either at most (float32 sums of keys may round the other way, rarely)
    assert (got[:n] - want).norm() / want.norm() <= 2 * 2.0 ** -9
    worst = (got[:n] - want).abs().amax(1) / want.pow(2).mean(1).sqrt()
    assert worst.max() <= 16 * 2.0 ** -9                   # every row, its largest channel four times its mean


def test_a_recorded_model_follows_the_eager_one():
    """Prompts of one size class whose attention makes the heads' keys, beside a context and without, recorded and eagerly."""
    from minivllm_amd.config import EngineConfig
    from minivllm_amd.engine.executor import Executor
    from minivllm_amd.engine.step import SeqStep
    from minivllm_amd.models import config_from_dict, expected_tensors
    from minivllm_amd.weights.device_random import DeviceRandomSource
    latent = {"heads": 2, "dim": 128, "rot_dim": 64, "vdim": 128, "q_rank": 64, "kv_rank": 128, "scale": 0.07, "rot": {"dims": 64, "base": 1e4}}

    def executor(graphs):
        arch, cfg = config_from_dict({"architecture": "Dutilix", "vocab": 256, "width": 128, "norm": {"eps": 1e-5}, "torch_dtype": "bfloat16",
                                      "logit_scale": 1.0, "layers": [{"type": "latent_attention", "mixer": latent,
                                                                      "mlp": {"kind": "dense", "ff": 128}}] * 2})
        source = DeviceRandomSource(expected_tensors(arch, cfg), 1, torch.bfloat16, torch.device(DEV), std=0.08)
        return Executor(EngineConfig(model="", dtype="bfloat16", max_model_len=1024, max_num_batched_tokens=1024, max_num_batched_seqs=16,
                                     kv_cache_block_size=16, kv_cache_num_blocks=256, use_cuda_graph=graphs), model=(arch, cfg, source))
    recorded, eager = executor(True), executor(False)
    gen = torch.Generator().manual_seed(3)
    text = [torch.randint(0, 256, (700,), generator=gen).tolist() for _ in range(3)]
    tables = [list(range(44 * s, 44 * s + 44)) for s in range(3)]
    for turn in range(3):
        for cut in ([(100, 0)], [(97, 0)], [(60, 0), (45, 0)], [(90, 0), (1, 0), (14, 0)], [(100, 97)], [(99, 90)]):
            made = [SeqStep(tokens=text[s][start:start + q], start=start, block_tables=[tables[s]], state_slot=s, want=[q - 1])
                    for s, (q, start) in enumerate(cut)]
            got, plain = recorded.step(made).clone(), eager.step(made).clone()
            assert torch.equal(got, plain), cut                # (both choose by the step and its class, and add in the same orders)
    entries = [{e[0] for e in ledger} for ledger in recorded.graph_ledger.values()]
    assert entries and all("mv_attention_latent_heads" in e and "mv_attention_latent_prompt" not in e for e in entries)


@pytest.mark.parametrize("spread", [0.3, 1.0, 3.0])
@pytest.mark.parametrize("n, start", [(65, 0), (200, 0), (700, 0), (90, 500)])
def test_no_further_from_64_bits_than_the_latents_space(n, start, spread):
    """Both ways of the same attention, scores of three deviations. Whichever roundings one way has in place of the other's, its error
    is no larger (0.75 to 0.93 of it, measured over 65 to 8,000 tokens)."""
    from minivllm_amd.engine.step import AttentionPlan
    from minivllm_amd.kernels.ops import Ops, latent_operands
    from minivllm_amd.parts import Workspace
    R, dr, H, ps = 256, 64, 4, 16
    ops, gen, ctx, scale = Ops(torch.bfloat16), torch.Generator().manual_seed(n), n + start, 192 ** -0.5
    rand = lambda *shape: torch.randn(*shape, generator=gen)
    lat, q = rand(ctx, R + dr).bfloat16(), (rand(n, H * (128 + dr)) * spread).bfloat16()
    w_k, w_v = (rand(H, 128, R) / math.sqrt(R)).bfloat16(), (rand(H, 128, R) / math.sqrt(R)).bfloat16()
    angle = torch.arange(ctx)[:, None] * (1e4 ** (-torch.arange(0, dr, 2) / dr))[None]
    table = torch.cat([angle.cos(), angle.sin()], 1).float()
    want = torch.empty(n, H, 128, dtype=torch.float64)
    cos, sin = table[start:, :32].double(), table[start:, 32:].double()
    hidden = torch.arange(ctx)[None] > torch.arange(start, ctx)[:, None]
    for h in range(H):
        x, c = q.double().view(n, H, -1)[:, h], lat[:, :R].double()
        a, b = x[:, 128:160], x[:, 160:]
        s = x[:, :128] @ (c @ w_k[h].double().T).T + torch.cat([a * cos - b * sin, b * cos + a * sin], -1) @ lat[:, R:].double().T
        want[:, h] = torch.softmax((s * scale).masked_fill(hidden, -math.inf), -1) @ (c @ w_v[h].double().T)
    i32 = lambda x: torch.tensor(list(x), dtype=torch.int32, device=DEV)
    npages = -(-ctx // ps)
    pages = torch.zeros(npages, ps, R + dr, dtype=torch.bfloat16, device=DEV)
    pages.view(-1, R + dr)[:ctx] = lat.to(DEV)
    bt, positions, seq, cl, cu = i32(range(npages)).view(1, -1), i32(range(start, ctx)), i32([0] * n), i32([ctx]), i32([0, n])
    plan = AttentionPlan(decode_only=False, max_q_len=n, max_context_len=ctx, n_seqs=1, q_lens=[n], cu_seqlens=cu,
                         workspace=Workspace(torch.device(DEV)), starts=[start])
    blocks = -(-ctx // 32)
    scratch = lambda *shape: torch.empty(*shape, dtype=torch.bfloat16, device=DEV)
    k, v, kr, own, latent = scratch(blocks, H, 4096), scratch(blocks, H, 4096), scratch(blocks, 32 * dr), scratch(n, H * 128), scratch(n, H * 128)
    q, w_k, w_v, table = q.to(DEV), w_k.to(DEV), w_v.to(DEV), table.to(DEV)
    ops.latent_expand(pages, bt, ps, plan, cl, latent_operands(w_k), latent_operands(w_v), H, R, dr, blocks, k, kr, v)
    ops.attention_latent_heads(q, own, k, kr, v, plan, positions, seq, cl, H, dr, scale, table)
    qa, mixed = torch.empty(n, H, R + dr, device=DEV), torch.empty(n, H, R, device=DEV)
    ops.head_linear(q.unflatten(1, (H, 128 + dr)), w_k, qa, seq, tail=dr, table=table, positions=positions, w_rows=w_k.transpose(1, 2).contiguous())
    ops.attention_latent(qa, mixed, pages, bt, ps, positions, seq, H, R, dr, scale, plan=plan, pages_t=pages[:, :, :R].transpose(1, 2).contiguous())
    ops.head_linear(mixed, w_v.transpose(1, 2).contiguous(), latent, seq, w_rows=w_v)
    off = [float((o.double().cpu() - want.flatten(1)).norm() / want.norm()) for o in (own, latent)]
    assert off[0] <= off[1], off


@pytest.mark.parametrize("R, dr, H, lens, starts, surplus", [
    (256, 64, 2, [70, 1], [0, 40], 1),                     # an odd number of blocks
    (256, 64, 2, [70, 1], [0, 40], 3000),                  # grid shorter than the room
    (128, 64, 64, [66, 3, 1], [2400, 31, 700], 0),         # three and more turns of a workgroup
    (256, 0, 64, [66, 3, 1], [2400, 31, 700], 500)])
def test_keys_and_values_are_made_whatever_the_room(R, dr, H, lens, starts, surplus):
    """Every block that there is, its sums as float32 has them, and nothing behind the last: workgroups walk over the blocks."""
    from minivllm_amd.engine.step import AttentionPlan
    from minivllm_amd.kernels.ops import Ops, latent_operands
    ops, gen, ps = Ops(torch.bfloat16), torch.Generator().manual_seed(1), 16
    rand = lambda *shape: torch.randn(*shape, generator=gen)
    context = [q + s for q, s in zip(lens, starts)]
    pages_of = [-(-c // ps) for c in context]
    pages = rand(sum(pages_of), ps, R + dr).bfloat16().to(DEV)
    table, at = torch.zeros(len(lens), max(pages_of), dtype=torch.int32), 0
    for i, p in enumerate(pages_of):
        table[i, :p] = torch.arange(at, at + p)
        at += p
    w_k, w_v = ((rand(H, 128, R) / math.sqrt(R)).bfloat16().to(DEV) for _ in range(2))
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    plan = AttentionPlan(decode_only=False, max_q_len=max(lens), max_context_len=max(context), n_seqs=len(lens), q_lens=lens, starts=starts,
                         cu_seqlens=i32([0] + torch.tensor(lens).cumsum(0).tolist()))
    per = [-(-c // 32) for c in context]
    real, blocks = sum(per), sum(per) + surplus
    mark = lambda *shape: torch.full(shape, 7.0, dtype=torch.bfloat16, device=DEV)
    k, v, kr = mark(blocks, H, 4096), mark(blocks, H, 4096), mark(blocks, 32 * max(dr, 1))
    ops.latent_expand(pages, table.to(DEV), ps, plan, i32(context), latent_operands(w_k), latent_operands(w_v), H, R, dr, blocks, k, kr, v)
    slot = torch.arange(32)                                # (of a key in its block: tile, and place in the tile)
    tile, rho = slot // 4 % 2, 4 * (slot // 8) + slot % 4
    for i, c in enumerate(context):
        lat = torch.zeros(32 * per[i], R + dr, dtype=torch.bfloat16, device=DEV)
        lat[:c] = pages[table[i, :pages_of[i]].to(DEV).long()].reshape(-1, R + dr)[:c]
        first = sum(per[:i])
        # k [block, head, tile, 4 steps, 4 groups, 16 keys, 8]; v [block, head, 8 tiles, 4 groups of 8 keys, 16 channels, 8 keys]
        got_k = k[first:first + per[i]].view(-1, H, 2, 4, 4, 16, 8)[:, :, tile, :, :, rho]          # [32, block, head, step, group, 8]
        got_k = got_k.permute(1, 0, 2, 3, 4, 5).reshape(-1, H, 128)
        got_v = v[first:first + per[i]].view(-1, H, 8, 4, 16, 8).permute(0, 3, 5, 1, 2, 4).reshape(-1, H, 128)
        for got, w in ((got_k, w_k), (got_v, w_v)):
            want = (lat[:, :R].double().cpu() @ w.double().cpu().reshape(H * 128, R).T).view(-1, H, 128).to(DEV)
            assert bool(((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-5).all())
        if dr:
            got = kr[first:first + per[i]].view(-1, 2, dr // 32, 4, 16, 8)[:, tile, :, :, rho].permute(1, 0, 2, 3, 4).reshape(-1, dr)
            assert torch.equal(got, lat[:, R:])
    assert bool((k[real:] == 7).all()) and bool((v[real:] == 7).all()) and bool((kr[real:] == 7).all())


def test_one_recording_serves_the_contexts_of_its_class():
    """Recorded with few keys and replayed with many, and the other way: the bits of the eager step, whose rooms follow its own keys."""
    from minivllm_amd.config import EngineConfig
    from minivllm_amd.engine.executor import Executor
    from minivllm_amd.engine.step import SeqStep
    from minivllm_amd.models import config_from_dict, expected_tensors
    from minivllm_amd.weights.device_random import DeviceRandomSource
    latent = {"heads": 2, "dim": 128, "rot_dim": 64, "vdim": 128, "q_rank": 64, "kv_rank": 128, "scale": 0.07, "rot": {"dims": 64, "base": 1e4}}

    def executor(graphs):
        arch, cfg = config_from_dict({"architecture": "Dutilix", "vocab": 256, "width": 128, "norm": {"eps": 1e-5}, "torch_dtype": "bfloat16",
                                      "logit_scale": 1.0, "layers": [{"type": "latent_attention", "mixer": latent,
                                                                      "mlp": {"kind": "dense", "ff": 128}}] * 2})
        source = DeviceRandomSource(expected_tensors(arch, cfg), 1, torch.bfloat16, torch.device(DEV), std=0.08)
        return Executor(EngineConfig(model="", dtype="bfloat16", max_model_len=1024, max_num_batched_tokens=1024, max_num_batched_seqs=16,
                                     kv_cache_block_size=16, kv_cache_num_blocks=256, use_cuda_graph=graphs), model=(arch, cfg, source))
    recorded, eager = executor(True), executor(False)
    gen = torch.Generator().manual_seed(3)
    text = [torch.randint(0, 256, (1024,), generator=gen).tolist() for _ in range(2)]
    tables = [list(range(64 * s, 64 * s + 64)) for s in range(2)]

    def both(cut):
        made = [SeqStep(tokens=text[s][start:start + q], start=start, block_tables=[tables[s]], state_slot=s, want=[q - 1]) for s, q, start in cut]
        return recorded.step(made).clone(), eager.step(made).clone()
    for s in range(2):                                     # contexts that later steps follow, and rewrite with the same numbers
        for start in range(0, 1024, 512):
            both([(s, 512, start)])
    before = len(recorded._mixed_graphs)
    for order in (1, -1):
        for cut in [[(0, 100, 0)], [(0, 98, 31)], [(0, 112, 300)], [(0, 97, 927)], [(0, 112, 912)]][::order]:
            got, plain = both(cut)
            assert torch.equal(got, plain), cut
    assert len(recorded._mixed_graphs) == before + 1
    for cut in [[(0, 60, 0), (1, 45, 3)], [(0, 60, 900), (1, 45, 970)], [(0, 111, 913), (1, 1, 1023)]]:
        got, plain = both(cut)
        assert torch.equal(got, plain), cut
    assert len(recorded._mixed_graphs) == before + 2
    assert all("mv_attention_latent_heads" in {e[0] for e in ledger} for key, ledger in recorded.graph_ledger.items() if key[1] == 112)
