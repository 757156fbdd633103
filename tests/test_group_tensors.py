"""What a parameter group hands out is made in C++ (empty_list, strided_list of odc_torch.cpp): memory of its
own per gathered parameter, gradients that alias the published accumulation, the errors of torch's functions."""

import pytest
import torch

from helpers import assert_bit_equal
from odc_amd import _native


def test_arguments_are_checked():
    module = _native.load_torch_binding()
    for args in (([(2, 3)], "float32", 0), ([2], torch.float32, 0), ([(2, -3)], torch.float32, 0), ([(2,)], torch.float32)):
        with pytest.raises((TypeError, AssertionError)):
            module.empty_list(*args)
    base = torch.arange(24.0)[4:]
    (a, b) = module.strided_list(base, [((2, 3), (3, 1), 1), ((0, 5), (5, 1), 0)])
    assert torch.equal(a, base[1:7].view(2, 3)) and a.untyped_storage().data_ptr() == base.untyped_storage().data_ptr()
    assert b.shape == (0, 5)
    with pytest.raises(RuntimeError):
        module.strided_list(base, [((100, 3), (3, 1), 0)])  # leaves the storage
    for views in ([((2,), (1,))], [None], 5):
        with pytest.raises(TypeError):
            module.strided_list(base, views)
    with pytest.raises(TypeError):
        module.strided_list(None, [])


@pytest.mark.gpu
@pytest.mark.parametrize("param_dtype", [None, torch.bfloat16], ids=str)
@pytest.mark.parametrize("shapes", [[(8, 3), (16,)], [(7, 5, 2), (1,), (9, 4), (24, 2)]], ids=str)
def test_a_group_through_a_minibatch(make_world, shapes, param_dtype):
    from odc_amd.fsdp import fsdp2

    W = 8
    group = make_world(W, 1 << 20)
    fsdp2.patch_fsdp2()
    try:
        unit = fsdp2.ParamGroup(shapes, torch.float32, group, param_dtype=param_dtype, reduce_dtype=torch.float32)
        gen = torch.Generator().manual_seed(2)
        full = [torch.randn(s, generator=gen) for s in shapes]
        unit.load_full_params([f.cuda() for f in full])
        first, second = unit.unshard(), unit.unshard()
        dtype = param_dtype or torch.float32
        for a, b, f in zip(first, second, full):
            assert a.shape == f.shape and a.dtype == dtype and not a.requires_grad and a.is_contiguous()
            assert_bit_equal(a, f.to(dtype))
            b.zero_()  # memory of its own
            assert_bit_equal(a, f.to(dtype))
        assert len({t.untyped_storage().data_ptr() for t in first + second}) == 2 * len(shapes)

        grads = [torch.randn(s, generator=gen).to(dtype) for s in shapes]
        # gradients that are not contiguous are accumulated by value
        unit.reduce([torch.stack([g, g], -1)[..., 0].cuda() for g in grads])
        handed_out = unit.update_gradients()
        for p, (g, shape, got) in enumerate(zip(grads, shapes, handed_out)):
            rows = unit.local_shard_rows(p, 0)
            assert got.shape == (rows, *shape[1:])
            assert_bit_equal(got, g[:rows].float() / W)
            got.fill_(3.0)
            lo = unit.acc_offsets[p]
            assert (fsdp2.get_reduction_service().get_accumulation(id(unit))[lo : lo + got.numel()] == 3.0).all()
    finally:
        fsdp2.unpatch_fsdp2()


@pytest.mark.gpu
def test_out_of_memory_is_what_torch_raises():
    module = _native.load_torch_binding()
    with pytest.raises(torch.OutOfMemoryError):
        module.empty_list([(1 << 50,)], torch.float32, 0)
    (t,) = module.empty_list([(4, 2)], torch.float16, 0)
    assert t.shape == (4, 2) and t.dtype == torch.float16 and t.is_cuda
