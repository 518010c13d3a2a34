"""Layers like the ones before them, launched from a list.

A step that is not replayed as a graph (a prompt's portion, a mixed step) is launched kernel by kernel, and between two
launches of 4 us stand some 9 us of Python: parts that choose kernels, wrappers that check every tensor.  For a layer
like one that has just run (equal specs, the same step) all of that comes out the same, so a stretch of one or a few
layers is run once with its calls written down (`kernels.lib.Launches`) and the calls are made again for every
further stretch, the weights' and caches' addresses replaced by that stretch's.  Nothing outlives the step.

What one stretch leaves for the next (the pending output of its last part) lies in two sets of buffers in turn: the ones that the
written-down stretch read and the ones that it wrote.
"""

import torch

from atomserve_amd.kernels import ops
from atomserve_amd.kernels.lib import Launches
from atomserve_amd.parts.base import DeltaSum, SplitSums
from atomserve_amd.parts.block import PreNormBlock, TwoNormsBlock
from atomserve_amd.parts.norm import PendingRMSNorm

MOST_LAYERS = 4  # of a stretch
# Steps of more tokens are left alone: their kernels take longer than the host, and the buffers that a stretch holds are larger
# (Qwen3-0.6B sizes, the smallest model: 1,024 tokens take the GPU as long as the host).
MOST_TOKENS = 1024


def _plain(block) -> bool:
    """Whether the layer is of a kind whose launches may be written down, with nothing put in place of its methods."""
    return type(block) in (PreNormBlock, TwoNormsBlock) and "forward" not in vars(block) and all(
        "forward" not in vars(part) for part in block.parts().values())  # fmt: skip


def stretches(plan, blocks) -> tuple:
    """(first run, layers of a stretch, stretches after it) that covers the most runs, or None: runs from the first one on
    repeat the ones before them with equal specs, all writing caches of their own."""
    runs, best = plan.run, None

    def alike(i, j) -> bool:
        a, b = runs[i], runs[j]
        return (not a.reenter and not b.reenter and a.writes and b.writes and plan.cache_id(i) == i and plan.cache_id(j) == j
                and a.layer != b.layer and type(blocks[a.layer]) is type(blocks[b.layer])
                and blocks[a.layer].spec == blocks[b.layer].spec and not blocks[a.layer].cache_request()
                and (blocks[a.layer].parts().keys() == blocks[b.layer].parts().keys()))  # fmt: skip

    def follows(i):
        """What the run before `i` is told of the norm that comes."""
        norm = blocks[runs[i].layer].first_norm() if i < len(runs) else None
        return None if norm is None else (type(norm), norm.spec)

    for period in range(1, MOST_LAYERS + 1):
        for first in range(1, len(runs) - 2 * period + 1):
            count = 0
            while True:
                at = first + (count + 1) * period
                if at + period > len(runs) or follows(at + period) != follows(first + period) or not all(
                        alike(first + k, at + k) for k in range(period)):  # fmt: skip
                    break
                count += 1
            if count and (best is None or count * period > best[1] * best[2]):
                best = (first, period, count)
    return best


def _view_addresses(view, into: list) -> None:
    """The addresses of a cache view's tensors, or of a dict of views, in an order that equal kinds share."""
    if isinstance(view, dict):
        for name in sorted(view):
            _view_addresses(view[name], into)
    elif view is not None:
        for name in type(view).__slots__:
            found = getattr(view, name)
            if isinstance(found, torch.Tensor):
                into.append(found.data_ptr())


def _own_names(model, first: int, period: int) -> list:
    """For each run of the stretch that starts at run `first` the (part, attribute, has a copy) that are a layer's own
    tensors: all of its parts' attributes that are tensors or `ops.Streamed`."""
    return [[(name, attr, isinstance(v, ops.Streamed)) for name, part in model.blocks[model.plan.run[first + k].layer].parts().items()
             for attr, v in sorted(vars(part).items()) if isinstance(v, (torch.Tensor, ops.Streamed))] for k in range(period)]  # fmt: skip


def _own_addresses(model, step, names: list, start: int) -> list:
    """The addresses that belong to the stretch that starts at run `start`: its layers' tensors, its caches and the gains of
    the norms that follow its layers (which their last products may prepare)."""
    plan, found = model.plan, []
    for k, wanted in enumerate(names):
        i = start + k
        parts = model.blocks[plan.run[i].layer].parts()
        for name, attr, streamed in wanted:
            v = getattr(parts[name], attr)
            if streamed:
                found.append(v.rows.data_ptr())
                found.append(0 if v.wave is None else v.wave.data_ptr())
            else:
                found.append(v.data_ptr())
        _view_addresses(step.cache_view(plan.cache_id(i), True), found)
        after = model.blocks[plan.run[i + 1].layer].first_norm() if i + 1 < len(plan.run) else None
        if after is not None:
            found.extend(v.data_ptr() for _, v in sorted(vars(after).items()) if isinstance(v, torch.Tensor))
    return found


def _left(delta):
    """The tensors of a pending output, or None for a kind that is not handed on here."""
    if isinstance(delta, torch.Tensor):
        return [delta]
    if isinstance(delta, SplitSums):
        return [delta.sums]
    if type(delta) is PendingRMSNorm:
        return [delta.scaled, delta.ssq]
    if isinstance(delta, DeltaSum) and all(isinstance(p, torch.Tensor) for p in delta.parts):
        return list(delta.parts)
    return None


def run_again(model, made: Launches, step, before, after, first: int, period: int, count: int):
    """The `count` stretches after the one that starts at run `first`, whose launches `made` holds; before, after: the pending
    outputs that it took and gave.  Returns (runs done, the pending output); (0, after) if they are not its like."""
    taken, given = _left(before), _left(after)
    if not made.whole or taken is None or given is None or type(before) is not type(after) or \
            [(t.shape, t.dtype) for t in taken] != [(t.shape, t.dtype) for t in given]:  # fmt: skip
        return 0, after
    turns = [[t.data_ptr() for t in taken], [t.data_ptr() for t in given]]

    names = _own_names(model, first, period)
    made.aim(_own_addresses(model, step, names, first) + turns[0] + turns[1])
    done = 0
    for _ in range(count):
        start = first + done + period
        blocks = [model.blocks[model.plan.run[start + k].layer] for k in range(period)]
        if not all(_plain(b) for b in blocks):
            break
        targets = _own_addresses(model, step, names, start) + turns[1] + turns[0]
        if not made.fits(targets):
            break
        made.again(targets)
        turns.reverse()
        before, after = after, before
        done += period
    if done and type(after) is PendingRMSNorm:  # the norm that is pending is the next run's
        after = PendingRMSNorm(model.blocks[model.plan.run[first + period + done].layer].first_norm(), after.x, after.scaled, after.ssq)
    return done, after


def may_run_again(model, step, first: int, period: int) -> bool:
    """Whether the stretch that starts at run `first` is worth writing down in this step."""
    return (step.num_tokens <= MOST_TOKENS and not model.env.products.trials_pending()
            and not torch.cuda.is_current_stream_capturing()
            and all(_plain(block) and all(part.repeats(step) for part in block.parts().values())
                    for block in (model.blocks[model.plan.run[first + k].layer] for k in range(period))))  # fmt: skip
