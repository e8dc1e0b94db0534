"""Workspaces with room for the stage-engine kernels alone, and which kernel a workspace served last."""
from __future__ import annotations

import re

import pytest
import torch

from flashact_amd import _lib

# the owner word of a workspace (u32 at byte 20)
PI05_STAGE, MA2_STAGE, PI05_GROUP, MA2_GROUP = 2, 4, 6, 7


def owner(ws: torch.Tensor) -> int:
    return int(ws[20:24].view(torch.int32).item())


def zeroed(nbytes: int, device) -> torch.Tensor:
    raw = torch.zeros(nbytes + 256, dtype=torch.uint8, device=device)
    off = (-raw.data_ptr()) % 256
    return raw[off:off + nbytes]


def need(run, device) -> int:
    """Bytes of the stage-engine kernel for the request that ``run(workspace)`` launches: below them a
    request is refused with that number, and the groups, where they need more, are not taken."""
    with pytest.raises(_lib.FlashActError, match="workspace") as e:
        run(zeroed(256, device))
    return int(re.search(r"(?:required|needs) (\d+)", str(e.value)).group(1))
