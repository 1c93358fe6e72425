"""An installed package holds every library that importing it loads."""

import importlib.util
from pathlib import Path

from flash_lab import _hip

try:
    import tomllib
except ImportError:  # Python 3.10
    import tomli as tomllib

REPO = Path(__file__).resolve().parent.parent


def test_package_data_has_every_built_library():
    spec = importlib.util.spec_from_file_location(
        "flash_lab_csrc_build", REPO / "flash-attention-lab_amd" / "csrc" / "build.py"
    )
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    built = {build.OUTPUT.name, build.TORCH_OUTPUT.name}
    assert built == {_hip.LIB_NAME, _hip.TORCH_LIB_PATH.name}
    config = tomllib.loads((REPO / "pyproject.toml").read_text())
    assert built <= set(config["tool"]["setuptools"]["package-data"]["flash_lab"])
