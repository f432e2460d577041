"""The attention links: which pipelines they take, and which link a session of few tiles runs."""
import json
import shutil
from pathlib import Path

import numpy as np
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


class Recorder:
    """Device memory on the host; keeps the images that were loaded and the launches."""

    def __init__(self):
        self.images, self.launches, self.uploads = [], [], 0

    def current(self): pass
    def allocate(self, size, align=256): return 4096 * (1 + self.uploads)
    def free(self, addr): pass
    def zero(self, addr, size, stream=None): pass
    def upload(self, addr, data, stream=None): self.uploads += 1
    def synchronize(self, stream=None): pass
    def module_load(self, image): return self.images.append(image)
    def module_unload(self, module): pass
    def module_function(self, module, name, lds=0): return 1
    def launch(self, fn, params, grid, block, lds, stream=None): self.launches.append(grid[0])


def _open(link_json, tiles=4, **kw):
    """What a session of `tiles` tiles of 128 queries loads and launches: image bytes, workgroups."""
    from pipelink_amd.host.attention import open_session

    be = Recorder()
    q, kv = np.zeros((1, tiles, 128, 128), np.uint16), np.zeros((1, 1, 128, 128), np.uint16)
    open_session(link_json, q, kv, kv, backend=be, **kw).launch()
    return be.images[0], be.launches[0]


def test_few_tiles_run_the_half_tile_link_made_for_their_link_and_no_other(built, tmp_path):
    from pipelink_amd.pipec import linker

    cell = tmp_path / "cell"
    shutil.copytree(built, cell)
    link_json = cell / "link" / "link.json"
    assert _open(link_json) == ((cell / "half" / "link" / "pipeline.hsaco").read_bytes(), 8)
    assert _open(link_json, tiles=400) == ((cell / "link" / "pipeline.hsaco").read_bytes(), 400)
    # another mask in the pipeline and only the link redone: few tiles run it too, not what was linked before
    (cell / "pipeline.json").write_text(json.dumps(_pipeline(mask="fa.mask.window")))
    linker.link(cell / "pipeline.json", cell / "link")
    relinked = (cell / "link" / "pipeline.hsaco").read_bytes()
    assert relinked != (built / "link" / "pipeline.hsaco").read_bytes()
    assert _open(link_json, window=7) == (relinked, 4)
    fa_build.link_half(cell)   # and the half tiles of the new link, once asked for
    assert _open(link_json, window=7) == ((cell / "half" / "link" / "pipeline.hsaco").read_bytes(), 8)


def test_the_grid_is_of_the_tiles_of_the_link_that_is_opened(built):
    half = built / "half" / "link" / "pipeline.hsaco"
    assert _open(built / "half" / "link" / "link.json") == (half.read_bytes(), 8)
    assert _open(built / "half" / "link" / "link.json", tiles=400) == (half.read_bytes(), 800)
    assert _open(built / "half" / "link" / "link.json", image=half) == (half.read_bytes(), 8)


def test_a_link_may_be_handed_over_as_an_object(built):
    image = built / "link" / "pipeline.hsaco"
    link = json.loads((built / "link" / "link.json").read_text())
    assert _open(link, image=image) == (image.read_bytes(), 4) and _open(link, tiles=400, image=image) == (image.read_bytes(), 400)


# heads, S, window -> half tiles; the shapes that are not were measured slower with them (us half / whole in the comments)
@pytest.mark.parametrize("heads,s,window,half", [
    (128, 128, None, True), (192, 128, None, False), (32, 128 * 4, 64, True),                     # 0.96, 1.20, 0.79
    (128, 256, None, False), (45, 384, None, False), (51, 640, None, True), (32, 1024, None, True),  # 1.02, 1.07, 0.91, 0.86
    (28, 1152, 64, False), (32, 1152, 700, True), (35, 1152, 300, False), (42, 1152, 300, False),  # 1.05, 0.79, 1.15, 1.28
    (128, 384, None, False), (96, 512, None, False), (80, 512, 64, False), (76, 640, None, False),  # 1.16, 1.11, 1.24, 1.04
    (29, 1536, None, True), (12, 4096, None, True), (12, 4096, 300, False), (9, 3584, 942, False),  # 0.80, 0.79, 1.12, 1.11
    (32, 2048, None, False), (1, 4096, 1, True)])                                                 # 1.07, 0.7
def test_half_tiles_only_where_they_are_faster(heads, s, window, half):
    from pipelink_amd.host.attention import _half_tiles_pay

    assert _half_tiles_pay(heads, s, window) == half
