"""Decode graphs of sizes between the listed ones in groups of two ranks that share the GPU (tensor parallel with the custom
all-reduce inside the graphs, expert parallel with the exchange inside): the tokens are those of eager steps."""
import os
import socket
import tempfile

import pytest
import torch
import torch.multiprocessing as mp

pytestmark = pytest.mark.gpu


def _free_port():
    with socket.socket() as s:
        s.bind(("127.0.0.1", 0))
        return s.getsockname()[1]


def _prompts(n, seed):
    g = torch.Generator().manual_seed(seed)
    return [torch.randint(2, 512, (3 + i % 4,), generator=g).tolist() for i in range(n)]


def _worker(rank, world, port, out_dir, kind):
    os.environ.update(MASTER_ADDR="127.0.0.1", MASTER_PORT=str(port), MLOP_CUSTOM_AR="force")
    import torch.distributed as dist

    dist.init_process_group("gloo", rank=rank, world_size=world)
    torch.cuda.set_device(0)
    from mlopamd.models import build_model
    from mlopamd.models.config import get_config
    from mlopamd.parallel.comm import make_parallel_state
    from mlopamd.runtime.engine import Engine, EngineConfig
    from mlopamd.runtime.sampler import SamplingParams

    dev = torch.device("cuda", 0)
    cfg = get_config("tiny-llama" if kind == "tp" else "tiny-mixtral")
    full = build_model(cfg, device=dev, seed=4)
    ps = make_parallel_state(tp_size=2, ep_size=1) if kind == "tp" else make_parallel_state(tp_size=1, ep_size=world)
    shard = build_model(cfg, device=dev, pstate=ps, seed=4).load_shard_from(full)
    res = {}
    try:
        for key, graphs in (("eager", False), ("graph", True)):
            eng = Engine(shard, EngineConfig(max_num_seqs=64, max_num_batched_tokens=512, max_model_len=64, num_kv_blocks=160,
                                             use_graphs=graphs, graph_buckets=(32, 64)))
            res[key + "_sizes"] = sorted(eng.graphs)
            params = SamplingParams(max_tokens=6, ignore_eos=True)
            if kind == "ep":  # the smaller rank is padded to the agreed 48 rows
                res[key] = eng.generate(_prompts(40 if rank == 0 else 20, rank), params)
            elif ps.tp_rank == 0:
                res[key] = eng.generate(_prompts(40, 0), params)
                eng.shutdown()
            else:
                eng.worker_loop()
            res[key + "_steps"] = eng.stats["graph_steps"]
        res["error"] = ps.tp.car.error() if kind == "tp" else ps.ep.ex.error()
    finally:
        torch.cuda.synchronize()
        dist.barrier()
        if kind == "tp":
            ps.tp.car.close()
        elif ps.ep.ex is not None:
            ps.ep.ex.close()
        dist.destroy_process_group()
    torch.save(res, os.path.join(out_dir, f"r{rank}.pt"))


@pytest.mark.parametrize("kind", ["tp", "ep"])
def test_two_ranks_in_an_added_size(kind):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    d = tempfile.mkdtemp()
    mp.start_processes(_worker, args=(2, _free_port(), d, kind), nprocs=2, join=True, start_method="spawn")
    for r in range(2):
        res = torch.load(os.path.join(d, f"r{r}.pt"), weights_only=False)
        assert res["error"] == 0 and res["eager_sizes"] == [] and res["graph_sizes"] == [32, 48, 64]
        if kind == "ep" or r == 0:
            assert res["graph_steps"] > 0 and res["eager_steps"] == 0
            assert all(len(o) == 6 for o in res["graph"]) and res["graph"] == res["eager"]
