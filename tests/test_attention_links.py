"""The attention links: which pipelines they take, and which link a session of few tiles runs."""
import json
import shutil
from pathlib import Path

import pytest

from pipelink_amd.stages.attention import build as fa_build

pytestmark = pytest.mark.skipif(shutil.which("hipcc") is None and not Path("/opt/rocm/bin/hipcc").exists(), reason="needs the ROCm toolchain")


@pytest.fixture(scope="module")
def built(tmp_path_factory):
    out = tmp_path_factory.mktemp("attention")
    fa_build.build(out=out, one_unit=False)
    return out


def _pipeline(core="fa.core.plink", mask="fa.mask.causal"):
    """A pipeline file of the core and one mask, written without knowledge of the core's half tiles."""
    return {"pipelink_abi": {"schema": "3.0", "target": {"profile": "gfx950", "lto_arch": "amdgcn-amd-amdhsa--gfx950", "toolkit": "rocm-7.2.0"}},
            "pipeline": {"name": "mine", "stages": [{"artifact_path": core, "stage_id": "fa.core"}, {"artifact_path": f"{mask}.plink", "stage_id": mask}],
                         "handles": {"pipelink_fa_kv": {"class": "base", "binding": "bind", "domain": "smem", "owner": "claim:pipelink_fa_kv"}},
                         "phases": ["steady"], "exclusive": [], "domains": {"gmem_counter": {"capacity": 16}}, "depth_priority": [],
                         "regs_priority": [], "forced_bindings": {}, "topology": {"persistent": False, "scheduler": "static"}}}


@pytest.mark.parametrize("core,mfma", [("fa.core.plink", 64), ("fa.core_half.plink", 32)])
def test_a_pipeline_file_names_core_and_mask_and_nothing_of_their_inside(built, tmp_path, core, mfma):
    from pipelink_amd.pipec import linker

    for f in built.glob("*.plink"):
        shutil.copy(f, tmp_path / f.name)
    (tmp_path / "pipeline.json").write_text(json.dumps(_pipeline(core)))
    link = linker.link(tmp_path / "pipeline.json", tmp_path / "link")
    assert set(link["bindings"]) == {"pipelink_fa_kv"} and link["observed"]["mfma"] == mfma and link["observed"]["calls"] == 0
    assert [(e["stage_id"], e["bytes"]) for e in link["params"]["entries"]] == [("fa.core", 56), ("fa.mask.causal", 8)]
