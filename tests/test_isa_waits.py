"""The waits of the block-scaled GEMMs, checked on the gfx950 assembly that hipcc makes of
them (no GPU needed). Their stage buffers are filled by LDS-DMA under counted vmcnt waits
and handed over at bare s_barriers, so two things must hold on every path through the
compiled code, whatever loads the compiler deleted or moved: how many DMA operations can
still be in flight where a stage's data is read, and which LDS operations can still be
outstanding at a barrier."""
import os
import re
import shutil
import subprocess

import pytest

from miroxen_amd import build as hipbuild

CSRC = hipbuild.CSRC


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{(kernel, template arguments): [instruction or label, ..]} of blockscale.hip."""
    cc = hipbuild.hipcc()
    if shutil.which(cc) is None:
        pytest.skip("hipcc not available")
    out = str(tmp_path_factory.mktemp("isa") / "blockscale.s")
    flags = [f for f in hipbuild.HIPCC_FLAGS if f != "-shared"]
    subprocess.run([cc, *flags, "-I", os.path.join(hipbuild.ROOT, "include"), "-I", CSRC, "-S", "--cuda-device-only",
                    os.path.join(CSRC, "blockscale.hip"), "-o", out], check=True, capture_output=True)
    found, body = {}, None
    for line in open(out):
        m = re.match(r"_ZN\S*?\d((?:mxfp8|nvfp4)_gemm|gemm_ksplit)I(\S*?)EEv\S*:", line)
        if m:
            args = tuple(int(x) for x in re.findall(r"L[bi](\d+)", m.group(2)))
            body = found[m.group(1), args] = []
        elif line.startswith(".Lfunc_end"):
            body = None
        elif body is not None:
            s = line.split(";")[0].strip()
            if s and (s.startswith(".LBB") or not s.startswith(".")):
                body.append(s)
    return found


def _blocks(body):
    """Basic blocks [(instructions, successors)], block 0 the entry."""
    labels, blocks, cur = {}, [], []
    for s in body:
        if s.endswith(":"):
            if cur:
                blocks.append(cur)
            labels[s[:-1]], cur = len(blocks), []
        else:
            cur.append(s)
            if s.startswith(("s_cbranch", "s_branch", "s_endpgm")):
                blocks.append(cur)
                cur = []
    out = []
    for i, b in enumerate(blocks):
        last = b[-1].split()
        to = [] if last[0] == "s_endpgm" else [labels[last[1]]] if last[0].startswith(("s_branch", "s_cbranch")) else []
        if last[0] not in ("s_endpgm", "s_branch"):
            to.append(i + 1)
        out.append((b, to))
    return out


def _count(field, s):
    m = re.search(field + r"\((\d+)\)", s)
    return int(m.group(1)) if m else None


def _dma_in_flight(body, at):
    """For each instruction that starts with `at`, in program order: the most LDS-DMA
    operations that can be in flight there, over every path. Loads return in order, so
    vmcnt(n) leaves the n youngest; stores are left out (more seems in flight than is)."""
    blocks, worst, seen, todo = _blocks(body), {}, set(), [(0, "")]
    while todo:
        b, q = todo.pop()
        if (b, q) in seen:
            continue
        seen.add((b, q))
        code, to = blocks[b]
        for i, s in enumerate(code):
            if s.startswith("buffer_load") and s.split()[-1] == "lds":
                q += "D"
            elif s.startswith(("buffer_load", "global_load")):
                q += "L"
            elif s.startswith("s_waitcnt") and _count("vmcnt", s) is not None:
                n = _count("vmcnt", s)
                q = q[len(q) - n:] if n < len(q) else q
            if s.startswith(at):
                worst[b, i] = max(worst.get((b, i), 0), q.count("D"))
        q = q[-80:].lstrip("L")  # (what is older than the oldest DMA does not matter)
        todo += [(t, q) for t in to]
    return [worst[k] for k in sorted(worst)]


def _early(ni, nj):
    """DMA operations of a stage that mxfp8_gemm issues before the next stage begins."""
    sl, nd = ni * nj, 2 * (ni + nj)
    pre = 2 if sl >= 8 else 1
    return sum(sl + pre + u * 5 * sl // (4 * nd) < 2 * sl for u in range(nd))


MX = [(4, 4, 2), (4, 2, 3), (2, 2, 4)]


@pytest.mark.parametrize("ni,nj,nbuf", MX)
def test_mxfp8_stage_landed_at_its_barrier(kernels, ni, nj, nbuf):
    """Behind a stage barrier the next stage is read: in flight are at most the stages
    after it (nbuf - 2, and with two buffers the prefetch of later lines into LDS that
    nothing reads). Before stage 0 the ring is being filled: also the first operations of
    the last slot."""
    got = _dma_in_flight(kernels["mxfp8_gemm", (ni, nj, nbuf)], "s_barrier")
    stage = 2 * (ni + nj) * (nbuf - 2)
    assert got[0] <= stage + _early(ni, nj), got
    assert max(got[1:]) <= stage + (nbuf == 2), got


@pytest.mark.parametrize("f4,ni,nj,nb", [(f, *t) for f in (0, 1) for t in ((2, 2, 2), (2, 1, 3), (1, 1, 2))])
def test_ksplit_stage_landed_before_its_reads(kernels, f4, ni, nj, nb):
    """Every wave of gemm_ksplit has its own ring: where it reads a stage, at most the
    nb - 1 later ones are in flight."""
    for (name, args), body in kernels.items():
        if name == "gemm_ksplit" and args[:3] == (f4, ni, nj):
            assert args[4] == nb
            got = _dma_in_flight(body, "ds_read")
            assert got and max(got) <= 4 * (ni + nj) * (nb - 1), (args, got)


@pytest.mark.parametrize("ni,nj", [(4, 4), (4, 2), (2, 2)])
def test_nvfp4_stage_landed_at_its_barrier(kernels, ni, nj):
    assert max(_dma_in_flight(kernels["nvfp4_gemm", (ni, nj)], "s_barrier")) == 0


def _lds_outstanding(body):
    """For each s_barrier, in program order: the most LDS reads and writes that can be
    outstanding there, over every path (LDS operations return in order)."""
    blocks, worst, state, todo = _blocks(body), {}, {0: (0, 0)}, [0]
    while todo:
        b = todo.pop()
        n, (code, to) = list(state[b]), blocks[b]
        for i, s in enumerate(code):
            if s.startswith("ds_"):
                n[s.startswith("ds_write")] += 1
            if s.startswith("s_waitcnt") and _count("lgkmcnt", s) is not None:
                n = [min(x, _count("lgkmcnt", s)) for x in n]
            if s.startswith("s_barrier"):
                worst[b, i] = tuple(n)
        for t in to:
            old = state.get(t)
            new = tuple(min(max(x), 64) for x in zip(n, old or n))
            if new != old:
                state[t] = new
                todo.append(t)
    return [worst[k] for k in sorted(worst)]


def test_no_lds_read_outstanding_at_a_barrier(kernels):
    """Behind a barrier a slot that was read is filled again, or takes the output tile."""
    for name, body in kernels.items():
        got = _lds_outstanding(body)
        assert got and max(r for r, _ in got) == 0, (name, got)


def test_no_lds_write_outstanding_at_a_barrier(kernels):
    """Behind a barrier other waves read what was written (output tile, partial tiles)."""
    for name, body in kernels.items():
        got = _lds_outstanding(body)
        assert got and max(w for _, w in got) == 0, (name, got)
