"""Tile programs over tiles of several rows, cut short by the tensor's edge.

CPU: the kernel the plan emits, compiled for the host with a shim (one thread per lane, real
barriers, the shuffles through memory) and run on tensors lying between sentinels, so that a
read past a cut tile changes the result.  GPU: the same programs through the Handle.
"""

import ctypes
import hashlib
import re
import subprocess

import pytest
import torch

import ninetoothed_amd as ninetoothed
import ninetoothed_amd.language as ntl
from ninetoothed_amd import Symbol, Tensor

ROWS, WIDTH = Symbol("ROWS", constexpr=True), Symbol("WIDTH", constexpr=True)
CLANG = "/opt/rocm/llvm/bin/clang++"

SHIM = r"""
#include <pthread.h>
#include <algorithm>
#include <cmath>
#include <cstring>
#include <thread>
#include <vector>
#define __device__
#define __forceinline__ inline
#define __global__
#define __shared__ static
#define __launch_bounds__(n)
#define __restrict__
using std::max;
using std::min;
struct nt_dim { unsigned x; };
static thread_local nt_dim threadIdx;
static nt_dim blockIdx, gridDim;
static pthread_barrier_t nt_barrier;
static char nt_lane[256][16];
static void __syncthreads() { pthread_barrier_wait(&nt_barrier); }
template <typename T> T __shfl_xor(T v, int s, int) {  // every lane of the workgroup takes part
  T r;
  memcpy(nt_lane[threadIdx.x], &v, sizeof(T));
  __syncthreads();
  memcpy(&r, nt_lane[threadIdx.x ^ (unsigned)s], sizeof(T));
  __syncthreads();
  return r;
}
"""


def _host_kernel(source, tmp_path):
    """The emitted kernel as a host function run(void** args, grid)."""
    params = re.search(r"nt_generic_tile\((.*)\) \{\n", source).group(1).replace("__restrict__ ", "").split(", ")
    args = ", ".join(f"*({p.rsplit(' ', 1)[0]}*)a[{i}]" for i, p in enumerate(params))
    text = SHIM + source + f"""
extern "C" void run(void** a, unsigned grid) {{
  gridDim.x = grid;
  pthread_barrier_init(&nt_barrier, nullptr, 256);
  for (blockIdx.x = 0; blockIdx.x < grid; ++blockIdx.x) {{
    std::vector<std::thread> lanes;
    for (unsigned t = 0; t < 256; ++t) lanes.emplace_back([=] {{ threadIdx.x = t; nt_generic_tile({args}); }});
    for (auto& l : lanes) l.join();
  }}
  pthread_barrier_destroy(&nt_barrier);
}}
"""
    base = tmp_path / hashlib.sha256(text.encode()).hexdigest()[:16]
    base.with_suffix(".cpp").write_text(text)
    subprocess.run([CLANG, "-O0", "-std=c++17", "-w", "-shared", "-fPIC", "-pthread", f"{base}.cpp", "-o", f"{base}.so"],
                   check=True)
    return ctypes.CDLL(f"{base}.so").run


def _run_on_host(plan, values, tmp_path):
    source, grid, spec = plan.launch_spec(values)
    slots, keep = [], []
    for a in spec:
        if a[0] == "table":
            keep.append(a[1])
            slots.append(ctypes.c_void_p(a[1].ctypes.data))
        elif a[0] == "tensor":
            slots.append(ctypes.c_void_p(values[a[1]].data_ptr()))
        elif a[0] == "scalar":
            slots.append((ctypes.c_int64 if a[2] == "int64" else ctypes.c_float)(values[a[1]]))
        else:
            slots.append(ctypes.c_int64(a[1]))
    argv = (ctypes.c_void_p * len(slots))(*[ctypes.addressof(s) for s in slots])
    _host_kernel(source, tmp_path)(argv, ctypes.c_uint(grid))


# ----------------------------------------------------------------------- programs
def max_of_row_sums_application(x, out):
    out = ntl.max(ntl.sum(ntl.cast(x, ntl.float32), axis=1))  # noqa: F841


def sum_of_row_maxima_application(x, out):
    out = ntl.sum(ntl.max(ntl.cast(x, ntl.float32), axis=1))  # noqa: F841


def centred_application(x, out):
    x32 = ntl.cast(x, ntl.float32)
    out = x32 - ntl.sum(x32, axis=1)[:, None]  # noqa: F841


def _handle(kind):
    if kind == "centred":
        return ninetoothed.make(lambda x, o: (x.tile((ROWS, WIDTH)), o.tile((ROWS, WIDTH))), centred_application,
                                (Tensor(2), Tensor(2)))

    def arrangement(x, o):
        return x.tile((ROWS, WIDTH)).flatten(), o.tile((1,))

    application = max_of_row_sums_application if kind == "max_sum" else sum_of_row_maxima_application
    return ninetoothed.make(arrangement, application, (Tensor(2), Tensor(1)))


def _reference(kind, x, rows):
    """Per tile: a reduction of masked elements only is its identity."""
    x = x.double()
    if kind == "centred":
        return x - x.sum(1, keepdim=True)
    out = []
    for r0 in range(0, x.shape[0], rows):
        tile = x[r0:r0 + rows]
        past = rows - tile.shape[0]
        if kind == "max_sum":
            out.append(torch.cat([tile.sum(1), tile.new_zeros(past)]).max())
        else:
            out.append(torch.cat([tile.max(1).values, tile.new_full((past,), float("-inf"))]).sum())
    return torch.stack(out)


def _between_sentinels(shape, dtype, device):
    """Small whole numbers (every sum exact), all negative past the first row, 1000 on both sides."""
    n = shape[0] * shape[1]
    buf = torch.full((n + 64,), 1000.0, dtype=dtype, device=device)
    x = buf[32:32 + n].view(shape)
    x.copy_(-(torch.arange(n, device=device) % 3 + 1).view(shape))
    x[0] = 1
    return x


CASES = ((6, 64, 4), (3, 256, 2), (19, 40, 8), (6, 255, 4), (5, 17, 3), (9, 8, 7), (2, 1025, 3))


def _check(kind, rows, cols, tile, dtype, device, call):
    x = _between_sentinels((rows, cols), dtype, device)
    programs = -(-rows // tile)
    size = (rows, cols) if kind == "centred" else (programs,)
    buf = torch.full((int(torch.tensor(size).prod()) + 64,), 7.0, dtype=torch.float32, device=device)
    out = buf[32:-32].view(size)
    call(_handle(kind), x, out)
    ref = _reference(kind, x.cpu(), tile)
    assert torch.equal(out.cpu().double(), ref), (out, ref)
    assert (buf[:32] == 7.0).all() and (buf[-32:] == 7.0).all()


@pytest.mark.parametrize("dtype", (torch.float32, torch.bfloat16))
@pytest.mark.parametrize("kind", ("max_sum", "sum_max", "centred"))
@pytest.mark.parametrize("rows, cols, tile", CASES)
def test_cut_rows_on_the_host(rows, cols, tile, kind, dtype, tmp_path):
    def call(handle, x, out):
        names = handle._abi["public_args"]
        values = dict(zip(names, (x, out)))
        plan = handle._kernel.specialize(values, {"ROWS": tile, "WIDTH": cols})
        _run_on_host(plan, values, tmp_path)

    _check(kind, rows, cols, tile, dtype, "cpu", call)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", (torch.float32, torch.bfloat16, torch.float64))
@pytest.mark.parametrize("kind", ("max_sum", "sum_max", "centred"))
@pytest.mark.parametrize("rows, cols, tile", CASES + ((1001, 2048, 8), (333, 333, 5)))
def test_cut_rows(rows, cols, tile, kind, dtype):
    _check(kind, rows, cols, tile, dtype, "cuda", lambda handle, x, out: handle(x, out, ROWS=tile, WIDTH=cols))


def row_sum_application(x, out):
    out = ntl.sum(ntl.cast(x, ntl.float32))  # noqa: F841


def test_one_source_serves_every_stride(tmp_path):
    # Column tiles of tensors of any width: the element step is an argument of the kernel.  Unit
    # steps, which vectors need, and tiles of one element (any step) share a second one.
    handle = ninetoothed.make(lambda x, o: (x.tile((ROWS, 1)).flatten(), o.tile((1,))), row_sum_application,
                              (Tensor(2), Tensor(1)))
    sources = {}
    for width in (100, 101, 102, 128, 200, 333, 1):
        x = (torch.arange(64 * width) % 7).float().view(64, width)
        for v in (x, x.t().contiguous().t(), x[:1].expand(64, width)):
            out = torch.full((width,), 7.0)
            values = dict(zip(handle._abi["public_args"], (v, out)))
            plan = handle._kernel.specialize(values, {"ROWS": 64})
            sources.setdefault(plan.sources_for(values)[0], []).append((v, out, values, plan))
    assert len(sources) == 2
    for v, out, values, plan in [calls[i] for calls in sources.values() for i in (0, 1, -1)]:
        _run_on_host(plan, values, tmp_path)
        assert torch.equal(out, v.sum(0))


def centred_in_place_application(x):
    x = x - ntl.sum(x)  # noqa: F841


@pytest.mark.parametrize("width, whole_workgroup", ((16379, True), (16380, False), (16383, False)))
def test_lds_of_a_whole_workgroup_reduction_is_counted(width, whole_workgroup):
    # The stored tile, the sum and (where they fit beside them) the four waves' sums: 64 KiB at most.
    handle = ninetoothed.make(lambda x: (x.tile((1, WIDTH)),), centred_in_place_application, (Tensor(2),))
    plan = handle._kernel.specialize({"x": torch.empty(3, width)}, {"WIDTH": width})
    declared = sum(4 * int(n) for n in re.findall(r"__shared__ float \w+\[(\d+)\]", "\n".join(plan.decls)))
    assert declared == plan.lds_bytes <= 64 * 1024
    assert ("red0_w" in "\n".join(plan.decls)) == whole_workgroup


@pytest.mark.parametrize("x, vectors", ((torch.empty(6, 64), True), (torch.empty(6, 70)[:, 3:67], False),
                                        (torch.empty(64, 6).t(), False)))
def test_vectors_only_without_tables(x, vectors):
    # Tiles of several rows of a wider or transposed tensor keep their tables, and with them one
    # lane an element: lanes that took vectors would read a table's entries apart from each other.
    handle = _handle("centred")
    values = dict(zip(handle._abi["public_args"], (x, torch.empty(6, 64))))
    plan = handle._kernel.specialize(values, {"ROWS": 4, "WIDTH": 64})
    body = plan.sources_for(values)[0].split("nt_generic_tile(")[1]
    assert ("nt_ldv" in body) == ("nt_stv" in body) == vectors
