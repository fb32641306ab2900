"""Fast autoregressive sampler vs the plain sampler and the oracle rule."""
import numpy as np
import pytest
import torch

from oracle import convnet as ocn
from oracle import samplers as osa
from tests.conftest import gpu_banner
from tests.test_gpu_convnet import _machine, _oracle_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('shape,depth,C,act,prec,B', [((6, 5), 3, 32, 'elu', 'bf16', 70),
                                                     ((4, 4), 2, 32, 'relu', 'fp32', 33),
                                                     ((10, 10), 4, 32, 'relu', 'bf16', 48),
                                                     ((5, 7), 3, 64, 'elu', 'fp32', 20),
                                                     ((5, 7), 3, 64, 'elu', 'bf16', 20),
                                                     ((6, 6), 3, 48, 'relu', 'bf16', 40),
                                                     ((4, 5), 2, 24, 'elu', 'fp32', 30),
                                                     ((10, 10), 3, 32, 'relu', 'fp16', 40),
                                                     ((5, 6), 2, 64, 'elu', 'fp16', 17),
                                                     # rows of 11-16 pixels (two staging batches, > 64 KB
                                                     # of LDS), 17 pixels (per-pixel vertical pass), depth 20
                                                     ((4, 13), 3, 32, 'elu', 'fp16', 20),
                                                     ((3, 16), 4, 32, 'relu', 'bf16', 17),
                                                     ((3, 17), 3, 32, 'relu', 'bf16', 16),
                                                     ((10, 10), 20, 32, 'relu', 'fp16', 32)])
def test_fast_equals_plain_given_uniforms(rng, shape, depth, C, act, prec, B):
    """Same uniforms -> the same draws as AutoregressiveSampler (identical
    arithmetic), and the conditionals it drew from equal the full forward's."""
    import flowket_amd as fk
    gpu_banner(f'fast sampler shape={shape} depth={depth} C={C} {act} {prec} B={B}')
    m = _machine(shape, depth, C, act, prec, bias_scale=0.4)
    u = rng.random((B,) + shape)
    plain = next(fk.AutoregressiveSampler(m, B, uniforms=u))
    fs = fk.FastAutoregressiveSampler(m, B, uniforms=u)
    fs.keep_cond_logp = True
    fast = next(fs)
    assert torch.equal(plain, fast)
    full = m.conditional_log_probs(fast)
    got = fs.last_cond_logp.reshape(full.shape)
    assert torch.equal(got, full)


def test_fast_matches_oracle_rule_fp32(rng):
    import flowket_amd as fk
    gpu_banner('fast sampler fp32 vs oracle rule 5x4')
    m = _machine((5, 4), 3, 32, 'elu', 'fp32', bias_scale=0.5)
    B = 128
    u = rng.random((B, 5, 4))
    got = next(fk.FastAutoregressiveSampler(m, B, uniforms=u)).cpu().numpy().astype(np.float64)
    params = _oracle_params(m)
    ref = osa.ar_sample(lambda x: ocn.conditional_log_probs(params, x, 3, activation='elu'), u)
    lp = ocn.conditional_log_probs(params, ref, 3, activation='elu')
    margin = np.abs(np.exp(lp[..., 0]) - u).reshape(B, -1).min(axis=1)
    ok = margin > 1e-6
    assert ok.mean() > 0.9
    assert np.array_equal(got[ok], ref[ok])


def test_fast_sampler_chunks(rng):
    """mini_batch_size < batch_size draws in chunks with the same result."""
    import flowket_amd as fk
    gpu_banner('fast sampler chunked')
    m = _machine((4, 6), 2, 32, 'relu', 'bf16')
    u = rng.random((50, 4, 6))
    a = next(fk.FastAutoregressiveSampler(m, 50, uniforms=u))
    b = next(fk.FastAutoregressiveSampler(m, 50, mini_batch_size=16, uniforms=u))
    assert torch.equal(a, b)


@pytest.mark.parametrize('shape,depth,C,act,prec,B', [((5, 6), 4, 32, 'elu', 'fp16', 17),
                                                      ((3, 1), 5, 32, 'relu', 'bf16', 16),
                                                      ((1, 9), 5, 24, 'elu', 'fp16', 5),
                                                      ((4, 13), 10, 32, 'relu', 'fp16', 40),
                                                      ((3, 40), 9, 20, 'elu', 'bf16', 20),
                                                      ((6, 5), 12, 64, 'elu', 'bf16', 33),
                                                      ((4, 26), 6, 48, 'relu', 'fp16', 18),
                                                      ((3, 39), 4, 64, 'relu', 'bf16', 16),
                                                      ((7, 7), 20, 32, 'elu', 'bf16', 20),
                                                      ((4, 6), 10, 32, 'relu', 'fp32', 19),
                                                      ((3, 14), 5, 48, 'elu', 'fp32', 17),
                                                      ((3, 21), 9, 64, 'relu', 'fp32', 16)])
def test_workgroup_per_tile_equals_plain(rng, shape, depth, C, act, prec, B):
    """The workgroup-per-tile kernel: one to seven steps per super-tick (and a
    last super-tick that is not full), rows of one pixel, rows that the waves
    take in several groups, the widest rows the LDS holds, each kernel width
    and precision.  Draws and conditionals are those of the plain sampler, bit
    for bit."""
    test_fast_equals_plain_given_uniforms(rng, shape, depth, C, act, prec, B)


def _waves(shape, depth, C, prec, B):
    from flowket_amd import _lib
    code = {'fp32': _lib.FK_PREC_FP32, 'bf16': _lib.FK_PREC_BF16, 'fp16': _lib.FK_PREC_FP16}[prec]
    return _lib.load().fk_fast_sampler_waves(*shape, depth, C, code, B)


@pytest.mark.parametrize('shape,depth,C,act,prec,B,per_tile', [
    # three steps per super-tick, four times as many blocks or a few more (operands four steps old), each width
    ((4, 5), 7, 32, 'relu', 'fp16', 18, 4), ((3, 6), 8, 20, 'elu', 'bf16', 16, 4), ((4, 5), 7, 64, 'elu', 'bf16', 17, 4),
    ((3, 6), 8, 48, 'relu', 'fp16', 20, 4), ((4, 5), 7, 32, 'elu', 'fp32', 16, 4), ((3, 6), 8, 24, 'relu', 'fp32', 19, 4),
    # the widest rows that the LDS holds, and one pixel more
    ((3, 63), 7, 32, 'relu', 'fp16', 20, 4), ((3, 64), 9, 32, 'elu', 'bf16', 20, 1), ((3, 34), 7, 64, 'relu', 'bf16', 17, 4),
    ((3, 35), 7, 64, 'relu', 'bf16', 17, 1), ((3, 34), 8, 32, 'elu', 'fp32', 18, 4), ((2, 35), 8, 32, 'elu', 'fp32', 18, 1),
    # rows of one pixel and of a few, where one wave is faster, and FP32 at 64 channels
    ((5, 1), 5, 64, 'elu', 'fp16', 20, 1), ((4, 1), 8, 32, 'relu', 'fp32', 18, 1), ((4, 2), 3, 20, 'elu', 'fp32', 16, 1),
    ((3, 2), 3, 40, 'relu', 'bf16', 16, 4), ((3, 4), 4, 64, 'elu', 'fp32', 17, 1)])
def test_kernel_by_network_equals_plain(rng, shape, depth, C, act, prec, B, per_tile):
    """The draws of either kernel are those of the plain sampler, bit for bit;
    per_tile waves draw 16 of them."""
    assert _waves(shape, depth, C, prec, B) == per_tile
    test_fast_equals_plain_given_uniforms(rng, shape, depth, C, act, prec, B)


@pytest.mark.parametrize('shape,depth,C,act,prec,rounds', [
    ((4, 4), 3, 32, 'relu', 'fp16', 2), ((3, 6), 3, 24, 'elu', 'bf16', 2), ((3, 3), 3, 64, 'relu', 'bf16', 2),
    ((2, 2), 5, 48, 'elu', 'fp16', 2), ((3, 8), 3, 32, 'relu', 'fp16', 4), ((2, 3), 5, 32, 'elu', 'fp32', 2), ((3, 5), 3, 32, 'relu', 'fp32', 2)])
def test_kernel_by_batch_equals_plain(rng, shape, depth, C, act, prec, rounds):
    """A batch of as many tiles as workgroups in ``rounds`` rounds over the chip
    is drawn by four waves a tile and a larger one by one wave, in the same
    workspace (chunks of the larger batch, and the rest of it)."""
    import flowket_amd as fk
    cu = torch.cuda.get_device_properties(0).multi_processor_count
    B = rounds * cu * 16
    assert _waves(shape, depth, C, prec, B) == 4 and _waves(shape, depth, C, prec, B + 1) == 1
    m = _machine(shape, depth, C, act, prec)
    total = B + 17 + 40
    u = rng.random((total,) + shape)
    plain = next(fk.AutoregressiveSampler(m, total, uniforms=u))
    assert torch.equal(next(fk.FastAutoregressiveSampler(m, total, uniforms=u)), plain)
    assert torch.equal(next(fk.FastAutoregressiveSampler(m, total, mini_batch_size=B + 17, uniforms=u)), plain)
    assert torch.equal(next(fk.FastAutoregressiveSampler(m, B, uniforms=u[:B])), plain[:B])
