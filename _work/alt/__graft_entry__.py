"""Driver entry points: build() compiles the gfx950 extensions in-tree;
smoke() runs one tiny decode of the flagship model on cuda:0."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.abspath(__file__))


def build() -> None:
    env = dict(os.environ, PYTORCH_ROCM_ARCH="gfx950")
    subprocess.run(
        [sys.executable, "setup.py", "build_ext", "--inplace"],
        cwd=ROOT, env=env, check=True)
    sys.path.insert(0, ROOT)
    import xllm_service_amd  # noqa: F401
    import xllm_service_amd.engine.engine  # noqa: F401
    import xllm_service_amd.models.llama  # noqa: F401


def smoke() -> None:
    sys.path.insert(0, ROOT)
    import torch
    assert torch.cuda.is_available(), "smoke() needs an MI355X"
    from xllm_service_amd import ops
    assert ops.HAS_EXT, "gfx950 HIP extension not built"
    from xllm_service_amd.engine.engine import LLMEngine
    from xllm_service_amd.engine.sampling import SamplingParams

    eng = LLMEngine("llama-3-8b", device="cuda:0", max_kv_blocks=2048, seed=0)
    prompt = torch.randint(0, eng.cfg.vocab_size, (64,)).tolist()
    out = eng.generate([prompt], SamplingParams(max_tokens=8, ignore_eos=True),
                       timeout_s=300.0)
    assert len(out[0]) == 8, f"smoke decode produced {out}"
    print("smoke OK:", out[0])


if __name__ == "__main__":
    build()
    if len(sys.argv) > 1 and sys.argv[1] == "smoke":
        smoke()
