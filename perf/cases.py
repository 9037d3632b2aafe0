"""The work this package is used for, as cases that can be timed and compared: the attention layers and the
block-sparse linear layer through their public classes, at the sizes of the package's own configurations (T2T-ViT
token grids, the Mixer-B channel MLP, the long-sequence and block-sparse attention benchmarks) and over the ranges
around them.

A case is a dict of plain values.  ``kind`` names the layer: 'sblocal' (SBLocalAttention), 'local' (LocalAttention),
'bsattn' (BlockSparseAttention), 'sbbs' (SBBlockSparseAttention), 'linear' (BlockSparseLinear).  ``train`` adds the
gradients of every input (and of the weight of a linear layer) to the pass.
"""
import math

import torch

import fly_amd

DEVICE = 'cuda:0'
DTYPES = {'fp32': torch.float32, 'bf16': torch.bfloat16, 'fp16': torch.float16}
# longest sequence the block-sparse attention layouts are made for; shorter ones use its upper left corner
MAX_SEQUENCE = 4096


def listed():
    return [
        # one image through the second T2T attention layer with the window of 12 and 6 features its configuration asks
        # for: the smallest call, serving latency
        dict(name='sblocal_one_image_fp32', kind='sblocal', dtype='fp32', train=False, B=1, H=1, L=784, E=64,
             window=12, features=6, temp_dim=576, scale=1.0, padded=False),
        # the headline forward: two images on the 56 x 56 token grid, window 512, 128 features
        dict(name='sblocal_headline_fp32', kind='sblocal', dtype='fp32', train=False, B=2, H=1, L=3136, E=64,
             window=512, features=128, temp_dim=64, scale=64 ** -0.25, padded=False),
        # training the first T2T attention layer on a batch of 64 images
        dict(name='sblocal_t2t_train_fp32', kind='sblocal', dtype='fp32', train=True, B=64, H=1, L=3136, E=64,
             window=256, features=128, temp_dim=147, scale=1.0, padded=False),
        # a long document, 16 heads: inference in bfloat16, and the training step of the same layer
        dict(name='sblocal_long_bf16', kind='sblocal', dtype='bf16', train=False, B=1, H=16, L=16384, E=64,
             window=1024, features=256, temp_dim=64, scale=64 ** -0.25, padded=False),
        dict(name='sblocal_long_train_bf16', kind='sblocal', dtype='bf16', train=True, B=1, H=16, L=16384, E=64,
             window=1024, features=256, temp_dim=64, scale=64 ** -0.25, padded=False),
        # plain local attention in the first T2T layer (window 98), training in the model's own float32
        dict(name='local_t2t_train_fp32', kind='local', dtype='fp32', train=True, B=64, H=1, L=3136, E=64,
             window=98, temp_dim=147, scale=1.0, padded=False),
        # plain local attention over the long document, mixed-precision training, sequence of odd length in a padded batch
        dict(name='local_long_train_bf16', kind='local', dtype='bf16', train=True, B=2, H=12, L=10007, E=64,
             window=1024, temp_dim=64, scale=1.0, padded=True),
        # block-sparse attention (band and butterfly blocks), 12 heads of 4096 tokens: inference, and a training step
        # with the constructor's default attention dropout
        dict(name='bsattn_forward_bf16', kind='bsattn', dtype='bf16', train=False, B=8, H=12, L=4096, E=64,
             padded=False, dropout=0.0),
        dict(name='bsattn_train_dropout_bf16', kind='bsattn', dtype='bf16', train=True, B=8, H=12, L=4096, E=64,
             padded=False, dropout=0.1),
        # Scatterbrain on a block-sparse support (window and global blocks), training the first T2T layer
        dict(name='sbbs_t2t_train_fp32', kind='sbbs', dtype='fp32', train=True, B=64, H=1, L=3136, E=64, block=32,
             features=32, scale=64 ** -0.25),
        # the block-sparse linear of the Mixer-B channel MLP: training its widening layer on a batch of 256 images, and
        # one image through the narrowing layer
        dict(name='linear_widening_train_bf16', kind='linear', dtype='bf16', train=True, tokens=256 * 196,
             n_in=768, n_out=3072, bias=False),
        dict(name='linear_one_image_bf16', kind='linear', dtype='bf16', train=False, tokens=196, n_in=3072,
             n_out=768, bias=True),
    ]


def _log_uniform(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(['sblocal', 'sblocal', 'sblocal', 'local', 'local', 'bsattn', 'bsattn', 'sbbs', 'linear', 'linear'])
    train = rng.random() < 0.5
    if kind == 'linear':
        n_in, n_out = rng.choice([(768, 3072), (3072, 768), (512, 2048), (1024, 4096), (4096, 1024), (768, 768)])
        return dict(kind=kind, dtype=rng.choice(['bf16', 'bf16', 'fp16']), train=train,
                    tokens=_log_uniform(rng, 49, 50176 * 3145728 // max(3145728, n_in * n_out)), n_in=n_in, n_out=n_out,
                    bias=rng.random() < 0.5)
    if kind == 'bsattn':
        L = _log_uniform(rng, 250, 4096)
        padded = rng.random() < 0.3
        dropout = 0.1 if train and not padded and rng.random() < 0.5 else 0.0
        if dropout:
            L = max(256, L // 32 * 32)
        B = _log_uniform(rng, 1, 8)
        return dict(kind=kind, dtype=rng.choice(['bf16', 'bf16', 'fp16']), train=train, B=B, H=12, L=L, E=64,
                    padded=padded, dropout=dropout)
    if kind == 'sbbs':
        block = rng.choice([16, 32])
        L = _log_uniform(rng, 196, 3136) // block * block
        return dict(kind=kind, dtype=rng.choice(['fp32', 'fp32', 'bf16']), train=train, B=_log_uniform(rng, 1, 64), H=1,
                    L=L, E=64, block=block, features=rng.choice([16, 32, 64, 128]), scale=64 ** -0.25)
    # bands: images (many short sequences of one head) or documents (few long sequences of several heads); at most as
    # many rows as the largest listed case, which is 64 images of 3136 tokens or one document of 16 heads
    if rng.random() < 0.6:
        H, L = 1, _log_uniform(rng, 196, 3136)
        B = _log_uniform(rng, 1, 64)
        dtype = rng.choice(['fp32', 'fp32', 'bf16'])
        temp_dim, scale = rng.choice([147, 576]), 1.0
    else:
        H, L = rng.choice([4, 8, 12, 16]), _log_uniform(rng, 1000, 16384)
        B = max(1, min(4, 196608 // (H * L)))
        dtype = rng.choice(['fp32', 'bf16', 'bf16'])
        temp_dim, scale = 64, 64 ** -0.25
    case = dict(kind=kind, dtype=dtype, train=train, B=B, H=H, L=L, E=rng.choice([64, 64, 64, 32]),
                window=_log_uniform(rng, 12, 1024 if H > 1 else 512), temp_dim=temp_dim, scale=scale,
                padded=rng.random() < 0.25)
    if kind == 'sblocal':
        case['features'] = rng.choice([_log_uniform(rng, 6, 128), 128, 256 if H > 1 else 64])
    return case


class WindowAndGlobal:
    """One head's layout of a window of one block to each side, and a global block-row and block-column."""

    def __init__(self, block):
        self.block = block

    def make_layout(self, seqlen):
        r = torch.arange(seqlen // self.block)
        layout = ((r.view(-1, 1) - r.view(1, -1)).abs() <= 1).long()
        layout[:, 0] = 1
        layout[0, :] = 1
        return layout.unsqueeze(0)


class BandAndButterfly:
    """A band of four blocks to each side and a flat butterfly of size 8 with two factors, the same for every head."""
    block = 32

    def __init__(self, heads):
        self.heads = heads

    def make_layout(self, seqlen):
        r = torch.arange(seqlen // self.block)
        band = (r.view(-1, 1) - r.view(1, -1)).abs() <= 4
        butterfly = fly_amd.FlatBlockButterflySparsityConfig(8, 2, self.block).make_layout(seqlen) > 0
        return (band | butterfly).long().unsqueeze(0).repeat(self.heads, 1, 1)


def _butterfly_linear():
    return fly_amd.FlatBlockButterflySparsityConfig(8, 2, block=32)


def prepare(case, seed):
    """The layer a user's program keeps, and fresh inputs for it."""
    dtype = DTYPES[case['dtype']]
    train = case['train']
    g = torch.Generator(DEVICE).manual_seed(seed)
    torch.manual_seed(seed)

    def normal(*shape, scale=1.0):
        return (torch.randn(*shape, generator=g, device=DEVICE) * scale).to(dtype)

    state = dict(case=case, seed=seed)
    if case['kind'] == 'linear':
        layer = fly_amd.BlockSparseLinear(case['n_in'], case['n_out'], _butterfly_linear(), bias=case['bias'])
        layer = layer.to(DEVICE).to(dtype)
        state.update(layer=layer, x=normal(case['tokens'], case['n_in']).requires_grad_(train))
        if train:
            state['grad'] = normal(case['tokens'], case['n_out'])
        return state

    B, H, L, E = case['B'], case['H'], case['L'], case['E']
    scale = case.get('scale', 1.0)
    q, k, v = normal(B, L, H, E, scale=scale), normal(B, L, H, E, scale=scale), normal(B, L, H, E)
    if case['kind'] == 'sblocal' and H > 1:
        loud = torch.rand(L, generator=g, device=DEVICE) < 0.05      # a few keys stand out, as in trained attention
        k[:, loud] *= 4
    if case['kind'] == 'sblocal':
        layer = fly_amd.SBLocalAttention(case['window'], dim_heads=E, nb_features=case['features'],
                                         softmax_temp=case['temp_dim'] ** -0.5)
    elif case['kind'] == 'local':
        layer = fly_amd.LocalAttention(case['window'], softmax_temp=case['temp_dim'] ** -0.5)
    elif case['kind'] == 'bsattn':
        layer = fly_amd.BlockSparseAttention(BandAndButterfly(H), attention_dropout=case['dropout'],
                                             max_seq_length=MAX_SEQUENCE)
    else:
        layer = fly_amd.SBBlockSparseAttention(WindowAndGlobal(case['block']), dim_heads=E, nb_features=case['features'],
                                               max_seq_length=L)
    layer = layer.to(DEVICE).train(train)
    if case['kind'] in ('sblocal', 'sbbs'):
        layer.feature_map.new_feature_map(torch.device(DEVICE))       # the random projection, drawn once
        layer.feature_map.freeze_projection()
    mask = None
    if case.get('padded'):
        lengths = torch.randint(L // 2, L + 1, (B,), generator=g, device=DEVICE)
        lengths[0] = L
        mask = fly_amd.LengthMask(lengths, max_len=L)
    state.update(layer=layer, mask=mask, qkv=[x.requires_grad_(train) for x in (q, k, v)])
    if train:
        state['grad'] = normal(B, L, H, E)
    return state


def run(state):
    case, layer = state['case'], state['layer']
    if case['kind'] == 'linear':
        inputs = (state['x'],) + ((layer.weight,) + ((layer.bias,) if layer.bias is not None else ()) if case['train'] else ())
        with torch.set_grad_enabled(case['train']):
            out = layer(state['x'])
    else:
        inputs = state['qkv']
        options = {} if state['mask'] is None else dict(key_padding_mask=state['mask'])
        if case.get('dropout'):
            torch.manual_seed(state['seed'])          # the layer draws its dropout seed from this generator
        with torch.set_grad_enabled(case['train']):
            out, _ = layer(*inputs, **options)
    if not case['train']:
        return out
    return (out.detach(),) + torch.autograd.grad(out, inputs, state['grad'])


def _band_pairs(L, window):
    i = torch.arange(L)
    return int(((i + (window + 1) // 2).clamp(max=L) - (i - window // 2).clamp(min=0)).clamp(min=0).sum())


def work(case):
    """Each input read once and each output written once; products of the algorithm, two operations a multiply-add: forward
    scores and weighted values, backward the scores and value products again and the sums for the gradients."""
    size = 4 if case['dtype'] == 'fp32' else 2
    train = case['train']
    if case['kind'] == 'linear':
        nnz = int(_butterfly_linear().make_layout(case['n_out'], case['n_in']).sum()) * 32 * 32
        tokens = case['tokens']
        rows = tokens * (case['n_in'] + case['n_out'])
        return {'bytes': size * (rows + nnz) * (2 if train else 1), 'flops': 2 * tokens * nnz * (3 if train else 1)}
    B, H, L, E = case['B'], case['H'], case['L'], case['E']
    bytes_ = size * B * H * L * E * (8 if train else 4)
    m = 2 * (case.get('features', 0) // 2)
    if case['kind'] in ('sblocal', 'local'):
        pairs = B * H * _band_pairs(L, case['window'])
    else:
        block = 32 if case['kind'] == 'bsattn' else case['block']
        n = -(-L // block)
        if case['kind'] == 'bsattn':
            layout = BandAndButterfly(H).make_layout(MAX_SEQUENCE)[:, :n, :n]
        else:
            layout = WindowAndGlobal(block).make_layout(L)
        pairs = B * int(layout.sum()) * block * block
    forward = 2 * pairs * (2 * E + m) + 2 * B * H * L * (2 * E * (m // 2) + 2 * m * (E + 1))
    backward = 2 * pairs * (5 * E + 3 * m) + 2 * B * H * L * (2 * E * (m // 2) * 2 + 4 * m * (E + 1))
    return {'bytes': bytes_, 'flops': forward + (backward if train else 0)}


def tolerance(case):
    """About four times what the passes are off from the same computation in float64 on the same inputs (2-norm; largest
    entry), measured over these ranges at up to 2000 tokens:
    float32 Scatterbrain layers 1.0e-5; 1.3e-4 (products of operands in bf16 pieces, "all keys minus the band"),
    float32 local attention 7e-7; 5e-6, bfloat16 3e-3; 5e-2, float16 3e-4; 2e-3."""
    if case['dtype'] == 'fp32':
        return {'rel': 3e-6, 'max': 4e-5} if case['kind'] == 'local' else {'rel': 4e-5, 'max': 6e-4}
    if case['dtype'] == 'fp16':
        return {'rel': 1.2e-3, 'max': 1e-2}
    return {'rel': 1e-2, 'max': 0.2}
