"""bench.py without a GPU: every workload the usage line names exists, every committed rocprofv3 summary that bench.py
reads its `traffic` figures from is there and parses, and a multi-GPU request is refused with a message."""
import os
import re
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
import bench  # noqa: E402


def test_forward_kernels_are_named_by_the_plan():
    name = lambda B, N, D=128: bench.prefill_kernel_name(bench.ask_plan(lambda lib, p: lib.vsp_attn_prefill_plan(B, 32, 8, N, N, D, 1, 0, p)), D, False)
    assert name(4, 2048) == "prefill_bf16_kernel<128, false, 4, 1, 0>" and name(1, 777) == "prefill_bf16_kernel<128, false, 2, 2, 1>"
    assert name(2, 2048) == name(1, 8192) == "prefill_bf16_pipe_kernel<false, false>" and name(4, 2048, 64) == "prefill_bf16_kernel<64, false, 4, 1, 0>"


def test_usage_line_names_every_workload():
    usage = re.search(r"--workload ([\w|]+)\]", bench.__doc__).group(1).split("|")
    assert sorted(usage) == sorted(bench.WORKLOADS)


def test_profiles_behind_the_traffic_figures_exist_and_parse():
    for key, (fname, kernels, algorithmic) in bench.PROFILE_OF.items():
        assert key in bench.WORKLOADS, key
        path = os.path.join(ROOT, "profiles", fname)
        assert os.path.exists(path), path
        text = open(path).read()
        assert f"--workload {key} " in text, (fname, "was not made by the workload it is filed under")
        t = bench.traffic_from_profile(key)
        assert t is not None, fname
        assert t["source"] == "profiles/" + fname and t["algorithmic_bytes"] == algorithmic
        # the counters see at least the compulsory traffic (reads can hit in cache: a loose lower bound) and no more
        # than an order of magnitude above it
        total = t["fetch_bytes"] + t["write_bytes"]
        assert 0.4 * algorithmic <= total <= 20 * algorithmic, (key, total, algorithmic)
        for k in kernels:
            assert k in text, (fname, k)


def _template_parameters():
    """Kernels of the sources: name -> number of template parameters."""
    found = {}
    for name in os.listdir(os.path.join(ROOT, "vesper_amd", "csrc")):
        if name.endswith(".hip"):
            src = open(os.path.join(ROOT, "vesper_amd", "csrc", name)).read()
            for params, kernel in re.findall(r"(?:template <([^>]*)>\s*)?__global__ void (?:__launch_bounds__\([^\n]*?\) )?(\w+)\(", src):
                found[kernel] = len(params.split(",")) if params else 0
    return found


def test_summaries_name_kernels_of_the_sources():
    # a summary made before a kernel was renamed, split or given other template parameters describes code that is not here
    have = _template_parameters()
    assert have["bwd_dkdv_bf16_kernel"] == 2 and have["prefill_bf16_kernel"] == 5 and have["proj_reduce_kernel"] == 1
    for fname in sorted(os.listdir(os.path.join(ROOT, "profiles"))):
        text = open(os.path.join(ROOT, "profiles", fname)).read()
        for kernel, args in re.findall(r"vsp::\(anonymous namespace\)::(\w+_kernel)(?:<([^>]*)>)?\(", text):
            assert kernel in have, (fname, kernel)
            assert have[kernel] == (len(args.split(",")) if args else 0), (fname, kernel, args)
    for key, (fname, kernels, _) in bench.PROFILE_OF.items():
        for k in kernels:
            assert any(k.split("<")[0] in name for name in have), (key, k)


def test_more_than_one_gpu_is_refused_with_a_message():
    r = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--gpus", "2"], capture_output=True, text=True, timeout=120)
    assert r.returncode != 0
    assert "one GPU" in (r.stdout + r.stderr) or "1 GPU" in (r.stdout + r.stderr) or "single" in (r.stdout + r.stderr).lower()
