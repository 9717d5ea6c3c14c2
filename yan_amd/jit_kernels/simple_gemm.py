"""fp32 GEMM entry point: `c = alpha * a @ b^T + beta * c`, written in place, returns None.

Same contract as the reference's `gemm_float_nt` (`yan/jit_kernels/simple_gemm.py:18-57`): `a` is `[m, k]` and `b` is
`[n, k]`, both stored with their FIRST dimension contiguous (what `get_col_major_tensor` returns; the reference
passes `ldA = m`, `ldB = n` without looking at the strides), `c` is `[m, n]` row-major, all fp32 on the current
device; `m % 128 == 0` and `n % 64 == 0`; the call is asynchronous on the current stream; `m == 0` or `n == 0` returns
at once. Argument order of the JIT kernel is the reference's: `(m, n, k, alpha, A, ldA, B, ldB, beta, C, ldC, stream)`.
The reference compiles one kernel with a fixed 128 x 64 tile (`keys={}`); here the tile is a key. Large problems run on the bf16
matrix cores, every number taken apart into three (gemm/simple_gemm_bf16x3.hpp): no further from the exact product than the fp32
matrix cores, which the others and what does not come apart still use.
"""
import functools

import torch

from .heuristics import get_best_float_config, get_float_bf16x3_config, get_split_k_float_config
from .host_calls import FLOAT, remember_call, repeat_call
from .split_k import SPLIT_K_WORKSPACE_BYTES, split_k_enabled, split_k_launch_failed, split_k_workspace
from .tuner import FrozenKeys, jit_tuner
from .utils import current_raw_stream, get_num_sms

includes = ('"gemm/simple_gemm.hpp"', )
template = """
// Templated args from Python JIT call
constexpr auto BLOCK_M = {BLOCK_M};
constexpr auto BLOCK_N = {BLOCK_N};

__return_code = static_cast<int>(gemm_nt<BLOCK_M, BLOCK_N>(m, n, k,
        alpha,
        static_cast<float const*>(A), ldA,
        static_cast<float const*>(B), ldB,
        beta,
        static_cast<float*>(C), ldC,
        stream));
"""

# K split over SPLIT_K workgroups per tile; the parts meet in `workspace` (launch_float_nt_split_k in gemm/simple_gemm.hpp).
split_k_template = """
// Templated args from Python JIT call
constexpr auto BLOCK_M = {BLOCK_M};
constexpr auto BLOCK_N = {BLOCK_N};
constexpr auto kSplitK = {SPLIT_K};

__return_code = static_cast<int>(yan::launch_float_nt_split_k<BLOCK_M, BLOCK_N, kSplitK>(m, n, k,
        alpha,
        static_cast<float const*>(A), ldA,
        static_cast<float const*>(B), ldB,
        beta,
        static_cast<float*>(C), ldC,
        stream, workspace, workspace_bytes));
"""

bf16x3_includes = ('"gemm/simple_gemm_bf16x3.hpp"', )
bf16x3_template = """
// Templated args from Python JIT call
constexpr auto BLOCK_M = {BLOCK_M};
constexpr auto BLOCK_N = {BLOCK_N};
constexpr auto kSplitK = {SPLIT_K};

__return_code = static_cast<int>(yan::launch_float_nt_bf16x3<BLOCK_M, BLOCK_N, kSplitK>(m, n, k,
        alpha,
        static_cast<float const*>(A), ldA,
        static_cast<float const*>(B), ldB,
        beta,
        static_cast<float*>(C), ldC,
        stream{WORKSPACE}));
"""

arg_defs = (('m', int), ('n', int), ('k', int),
            ('alpha', float),
            ('A', torch.float), ('ldA', int),
            ('B', torch.float), ('ldB', int),
            ('beta', float),
            ('C', torch.float), ('ldC', int),
            ('stream', torch.cuda.Stream))
split_k_arg_defs = arg_defs + (('workspace', torch.uint8), ('workspace_bytes', int))


@functools.lru_cache(maxsize=None)
def float_kernel_plan(m: int, n: int, num_cus: int):
    """(name, keys, arg_defs) of the JIT kernel a call with these sizes uses; needs no GPU."""
    block_m, block_n = get_best_float_config(m, n, num_cus)
    return 'gemm_float_nt', FrozenKeys({'BLOCK_M': block_m, 'BLOCK_N': block_n}), arg_defs


@functools.lru_cache(maxsize=None)
def float_split_k_plan(m: int, n: int, k: int, num_cus: int):
    """(name, keys, arg_defs) of the split-K kernel a call with these sizes uses, or None when K is not split
    (`get_split_k_float_config`); needs no GPU."""
    plan = get_split_k_float_config(m, n, k, num_cus)
    if plan is None:
        return None
    block_m, block_n, split_k = plan
    return 'gemm_float_nt_split_k', FrozenKeys({'BLOCK_M': block_m, 'BLOCK_N': block_n, 'SPLIT_K': split_k}), split_k_arg_defs


@functools.lru_cache(maxsize=None)
def float_bf16x3_plan(m: int, n: int, k: int, num_cus: int, may_split: bool = True):
    """(name, keys, arg_defs) of the kernel on the bf16 matrix cores a call with these sizes uses, or None
    (`get_float_bf16x3_config`); it takes a workspace where it splits K. Needs no GPU."""
    plan = get_float_bf16x3_config(m, n, k, num_cus, may_split)
    if plan is None:
        return None
    block_m, block_n, split_k = plan
    keys = FrozenKeys({'BLOCK_M': block_m, 'BLOCK_N': block_n, 'SPLIT_K': split_k, 'WORKSPACE': ', workspace, workspace_bytes' if split_k > 1 else ''})
    return 'gemm_float_nt_bf16x3' + ('_split_k' if split_k > 1 else ''), keys, split_k_arg_defs if split_k > 1 else arg_defs


def _leading_dim(x: torch.Tensor) -> int:
    """Distance in elements between consecutive k of a `[rows, k]` tensor whose rows are contiguous."""
    rows, k = x.shape
    assert rows <= 1 or x.stride(0) == 1, 'a and b must have their first dimension contiguous (get_col_major_tensor)'
    ld = x.stride(1) if k > 1 else rows
    assert ld >= rows and ld % 4 == 0
    return ld


def gemm_float_nt(a: torch.Tensor, b: torch.Tensor, c: torch.Tensor,
                  alpha: float = 1.0, beta: float = 0.0) -> None:
    if repeat_call(FLOAT, alpha, a, b, beta, c):
        return
    m, k = a.shape
    n, k_ = b.shape
    m_, n_ = c.shape

    assert m % 128 == 0 and n % 64 == 0

    assert m == m_ and n == n_ and k == k_
    assert a.dtype == torch.float32 and b.dtype == torch.float32 and c.dtype == torch.float32
    assert c.is_contiguous()

    if m == 0 or n == 0:
        return

    ldA, ldB, ldC = _leading_dim(a), _leading_dim(b), n
    stream = current_raw_stream()
    args = (m, n, k, float(alpha), a, ldA, b, ldB, float(beta), c, ldC, stream)
    num_cus = get_num_sms()
    kernel_includes, code_template, workspace, workspace_token = includes, template, None, None
    plan = float_bf16x3_plan(m, n, k, num_cus, split_k_enabled())
    if plan is not None:
        name, keys, defs = plan
        kernel_includes, code_template = bf16x3_includes, bf16x3_template
        if defs is split_k_arg_defs:
            workspace, workspace_token = split_k_workspace(c.device, stream)
            args += (workspace, SPLIT_K_WORKSPACE_BYTES)
    else:
        name, keys, defs = float_kernel_plan(m, n, num_cus)
        split = float_split_k_plan(m, n, k, num_cus)
        if split is not None:
            workspace, workspace_token = split_k_workspace(c.device, stream)
            if workspace is not None:
                name, keys, defs = split
                code_template = split_k_template
                args += (workspace, SPLIT_K_WORKSPACE_BYTES)
    runtime = jit_tuner.compile_and_tune(name=name, keys=keys, space=(), includes=kernel_includes,
                                         arg_defs=defs, template=code_template, args=args)
    rc = runtime(*args)
    if rc != 0 and workspace_token is not None:
        split_k_launch_failed(workspace_token)
    assert rc == 0, f'{name} failed with HIP error {rc}'
    remember_call((FLOAT, float(alpha), a, b, float(beta), c), name, runtime, args, workspace)


def accuracy_test():
    """The reference's smoke check (`simple_gemm.py:59-73`): seed 42, 5120 x 2048 x 4096, against `a @ b.t()`."""
    from .utils import get_col_major_tensor
    torch.manual_seed(42)
    m, n, k = 5120, 2048, 4096
    a = torch.randn(m, k, dtype=torch.float32, device='cuda')
    b = torch.randn(n, k, dtype=torch.float32, device='cuda')
    c = torch.zeros(m, n, dtype=torch.float32, device='cuda')
    c_ref = a.double() @ b.double().t()
    gemm_float_nt(get_col_major_tensor(a), get_col_major_tensor(b), c)
    assert torch.allclose(c.double(), c_ref, rtol=1e-4, atol=1e-3)
    print('Simple GEMM test passed!')
