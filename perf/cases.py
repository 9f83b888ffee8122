"""The measured cases of the batched NES environment step: what a training or evaluation program has this framework
do, through its public entry points (rl.rlenv.RlEnv, rl.hostobs.RolloutStore and the C entry points bound by
rl.rlenv.bind_library), from a handful of consoles to two full rounds of waves.

A case's ``kind`` says which path it runs:
  env       one decision of a batch: the actions copied in, RlEnv.step, and with ``pack6`` the pictures packed on the
            device (rl_pack6)
  rollout   one decision drawn into the rollout store's ring, packed and copied to its pinned host row
  minibatch the learner's side of the store: two minibatches gathered from pinned host memory and unpacked
  smb       the SMB reward tracker over T steps of N envs, from the 15 RAM bytes it reads (rl10_smb_run)
  tracker   a game's reward tracker over the whole RAM of T x N env-steps (rl10_run)
"""
import ctypes
import math
import os
import sys
from pathlib import Path

import numpy as np
import torch

PKG = Path(__file__).resolve().parents[1] / 'ghostrun-lab_amd'
sys.path.insert(0, str(PKG))

# Compiled translations of the carts are kept on disk, as bench.py keeps them; a folder that cannot be written only
# means that each process compiles its own.
_CACHE = PKG / 'csrc' / '_build' / 'jit_cache'
try:
    _CACHE.mkdir(parents=True, exist_ok=True)
    os.environ.setdefault('RLENV_JIT_CACHE', str(_CACHE))
except OSError:
    pass

from rl import synth  # noqa: E402
from rl.hostobs import PACKED_BYTES, RolloutStore  # noqa: E402
from rl.rlenv import FRAME_BYTES, GAMES, RlEnv, bind_library, hip_library  # noqa: E402

DEVICE = 'cuda:0'
PLAN = 16                      # decisions' actions held ready, taken in turn
ROM_SEED = 3                   # the carts are the games a program loads: fixed, while inputs and env seeds vary
# The game each board's cart is stepped as when it is alone; in a mixed batch the boards take GAMES in turn.
BOARDS = {
    'smb': lambda: synth.smb_like_cart(ROM_SEED),
    'nrom': lambda: synth.nrom_cart(ROM_SEED),
    'mmc1': lambda: synth.mmc1_cart(ROM_SEED),
    'uxrom': lambda: synth.uxrom_cart(ROM_SEED),
    'cnrom': lambda: synth.cnrom_cart(ROM_SEED),
    'mmc2': lambda: synth.mmc2_cart(ROM_SEED),
    'mmc3': lambda: synth.mmc3_cart(ROM_SEED, blocks=12, sub_blocks=8),
}
_roms = {}


def _rom(board):
    if board not in _roms:
        _roms[board] = BOARDS[board]()
    return _roms[board]


def listed():
    return [
        # a few consoles watched or evaluated, everything at RlEnv's defaults: latency and launches are all there is
        dict(name='env-smb-16', kind='env', boards='smb', envs=16, moves=True, idle=30, dropout=True, levels=0,
             end=0.0, pack6=False),
        # a small, ragged training batch below the size whose code is translated
        dict(name='env-nrom-500', kind='env', boards='nrom', envs=500, moves=True, idle=30, dropout=True, levels=0,
             end=1 / 500, pack6=False),
        # a quarter of the GPU
        dict(name='env-nrom-2048', kind='env', boards='nrom', envs=2048, moves=True, idle=30, dropout=True, levels=0,
             end=1 / 500, pack6=False),
        # the benchmark's headline configuration: raw pads, no dropout, no idle frames
        dict(name='env-nrom-8192', kind='env', boards='nrom', envs=8192, moves=False, idle=0, dropout=False, levels=0,
             end=0.0, pack6=False),
        # SMB training as the reference trains it: sticky moves, dropout, idle frames, episodes from saved level starts
        dict(name='env-smb-4096-levels', kind='env', boards='smb', envs=4096, moves=True, idle=30, dropout=True,
             levels=32, end=1 / 500, pack6=False),
        # a banked cart on the library's own kernels, odd count
        dict(name='env-mmc3-777', kind='env', boards='mmc3', envs=777, moves=True, idle=30, dropout=True, levels=0,
             end=1 / 500, pack6=False),
        # two rounds of waves of a banked cart, pictures packed on the device
        dict(name='env-mmc3-16384-pack6', kind='env', boards='mmc3', envs=16384, moves=False, idle=0, dropout=False,
             levels=0, end=0.0, pack6=True),
        # a multi-game batch, one game of every board, each on its own stream
        dict(name='env-mixed-6x1024', kind='env', boards='smb,mmc1,uxrom,cnrom,mmc2,mmc3', envs=1024, moves=True,
             idle=30, dropout=True, levels=0, end=1 / 500, pack6=False),
        # a rollout: pictures packed and stored in pinned host memory while the next decision runs
        dict(name='rollout-nrom-1024', kind='rollout', boards='nrom', envs=1024, rows=3, moves=True, idle=30,
             dropout=True, levels=0, end=1 / 500),
        # the learner's epoch over a stored rollout, two minibatches of it
        dict(name='minibatch-32x16', kind='minibatch', envs=96, rows=16, batch=32),
        # the reward of a recorded SMB rollout worked out again: the standalone tracker at the benchmark's size
        dict(name='smb-8192x1024', kind='smb', envs=8192, steps=1024),
        # a game's rewards replayed from recorded RAM
        dict(name='tracker-castlevania-2048x64', kind='tracker', game='castlevania', envs=2048, steps=64),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(['env'] * 7 + ['rollout', 'minibatch', 'smb', 'tracker'])
    if kind == 'minibatch':
        batch, rows = _log(rng, 4, 48), _log(rng, 2, 20)
        return dict(kind=kind, envs=2 * batch + rng.randint(0, 64), rows=rows, batch=batch)
    if kind == 'smb':
        return dict(kind=kind, envs=_log(rng, 64, 8192), steps=_log(rng, 8, 1024))
    if kind == 'tracker':
        return dict(kind=kind, game=rng.choice(sorted(TRACKED)), envs=_log(rng, 32, 2048), steps=_log(rng, 4, 64))
    raw = rng.random() < 0.3
    opts = dict(moves=not raw, idle=0 if raw else rng.choice([4, 30]), dropout=not raw,
                levels=0, end=rng.choice([0.0, 1 / 500, 1 / 100]))
    if kind == 'rollout':
        return dict(kind=kind, boards='nrom', envs=_log(rng, 16, 1024), rows=rng.randint(2, 5), **opts)
    boards = rng.choice(['smb', 'nrom', 'mmc3', 'mixed'])
    if boards == 'mixed':
        few = rng.sample(['smb', 'mmc1', 'uxrom', 'cnrom', 'mmc2', 'mmc3'], rng.randint(2, 6))
        return dict(kind=kind, boards=','.join(few), envs=_log(rng, 8, 1024), pack6=rng.random() < 0.3, **opts)
    if boards == 'smb' and rng.random() < 0.5:
        opts.update(levels=rng.choice([8, 32]), moves=True, idle=30, dropout=True, end=1 / 500)
    return dict(kind=kind, boards=boards, envs=_log(rng, 8, 16384 if boards == 'mmc3' else 8192),
                pack6=rng.random() < 0.3, **opts)


# ------------------------------------------------------------------------------------------------ env


def _env(case, seed):
    boards = case['boards'].split(',')
    games = dict(zip(GAMES, boards))
    kw = dict(seed=seed, sticky=True, idle_max=case['idle'], dropout=case['dropout'], pad_mode=not case['moves'],
              ram_hash=not case['moves'], end_prob=case['end'], level_cap=case['levels'],
              roms={g: _rom(b) for g, b in games.items()}, boot={g: bytes(4) for g in games})
    env = RlEnv({g: case['envs'] for g in games}, device=DEVICE, **kw)
    env.jit_wait()                       # a program that measures itself waits for its translated kernels
    return env


def _actions(case, n, seed):
    """Action rows taken in turn. Moves: a policy that mostly goes right (d-pad choices 2-4), without Start and Select;
    raw pads: any byte."""
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    rand = lambda k: torch.randint(0, k, (PLAN, n), generator=gen, device=DEVICE)  # noqa: E731
    if not case['moves']:
        return rand(256).to(torch.int16)
    pad = torch.where(rand(10) < 7, 2 + rand(3), rand(9))
    return (pad + 9 * rand(3) + 27 * rand(3)).to(torch.int16)


def _warm(env, plan, steps):
    env.start()
    for t in range(steps):
        env.actions.copy_(plan[t % PLAN])
        env.step()


def _prepare_env(case, seed):
    env = _env(case, seed)
    plan = _actions(case, env.n, seed)
    st = dict(env=env, plan=plan, t=0)
    _warm(env, plan, 4)
    if case['levels']:
        # level starts as a run has them some way in: the first level's saves stand in its slots (an arrival takes
        # about 100 decisions of this cart), and half of the new episodes begin from a saved one
        _warm(env, plan, 120)
        env.set_level_prob(0.5)
    names = ['obs', 'emph', 'reward', 'done', 'masks', 'timeline', 'pads', 'events', 'info', 'parts']
    if not case['moves']:
        names.append('ram_hash')
    if case['levels']:
        names += ['start_level', 'level_now', 'progress_now']
    st['out'] = {k: getattr(env, k) for k in names}
    if case.get('pack6'):
        st['packed'] = torch.empty(env.n * PACKED_BYTES, dtype=torch.uint8, device=DEVICE)
        st['out']['packed'] = st['packed']
    return st


def _ok(lib, rc):
    if rc != 0:
        raise RuntimeError(lib.rlenv_error().decode())


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def _stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def _run_env(st):
    env = st['env']
    env.actions.copy_(st['plan'][st['t'] % PLAN])
    env.step()
    if 'packed' in st:
        _ok(env.lib, env.lib.rl_pack6(_ptr(env.obs), _ptr(st['packed']), env.obs.numel(), _stream()))
    st['t'] += 1
    return st['out']


# ------------------------------------------------------------------------------------------------ rollout store


def _host_row(store, address, size):
    """A row of the store's pinned memory as an array, which keeps the store (and so the memory) alive."""
    block = (ctypes.c_uint8 * size).from_address(address)
    block.store = store
    return np.ctypeslib.as_array(block)


def _prepare_rollout(case, seed):
    env = _env(case, seed)
    plan = _actions(case, env.n, seed)
    _warm(env, plan, 2)
    env.drop_obs_buffers()
    store = RolloutStore(env.lib, case['rows'], env.n, DEVICE, 1)
    emph = torch.zeros(env.n, 4, 224, dtype=torch.uint8, device=DEVICE)
    rows = [_host_row(store, store.row_address(0, t), env.n * PACKED_BYTES) for t in range(case['rows'] + 1)]
    return dict(env=env, plan=plan, store=store, emph=emph, rows=rows, t=0)


def _run_rollout(st):
    env, store, t = st['env'], st['store'], st['t']
    env.actions.copy_(st['plan'][t % PLAN])
    env.bind_obs(store.target(t), st['emph'])
    env.step()
    store.commit(0, t)
    st['t'] = t + 1 if t + 1 < len(st['rows']) else 0
    return dict(row=st['rows'][t], emph=st['emph'], reward=env.reward, done=env.done, info=env.info)


def _prepare_minibatch(case, seed):
    lib = bind_library(hip_library())
    store = RolloutStore(lib, case['rows'], case['envs'], DEVICE, case['batch'])
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    for t in range(case['rows'] + 1):      # stored pictures: colour indices
        store.target(t).random_(0, 64, generator=gen)
        store.commit(0, t)
    perm = torch.randperm(case['envs'], generator=torch.Generator().manual_seed(seed))
    return dict(store=store, perm=perm, batch=case['batch'])


def _run_minibatch(st):
    b = st['batch']
    return [x for x in st['store'].minibatches(0, st['perm'][:2 * b], b)]


# ------------------------------------------------------------------------------------------------ trackers


def _prepare_smb(case, seed):
    n, t = case['envs'], case['steps']
    ram = synth.smb_ram15(seed, n, t)
    return dict(lib=bind_library(hip_library()), n=n, t=t, ram=torch.from_numpy(ram).to(DEVICE),
                state=torch.zeros(n, 80, dtype=torch.uint8, device=DEVICE),
                reward=torch.zeros(t, n, dtype=torch.float32, device=DEVICE),
                done=torch.zeros(t, n, dtype=torch.uint8, device=DEVICE))


def _run_smb(st):
    st['state'].zero_()
    _ok(st['lib'], st['lib'].rl10_smb_run(_ptr(st['ram']), st['t'], st['n'], 4, _ptr(st['state']), _ptr(st['reward']),
                                          _ptr(st['done']), _stream()))
    return dict(reward=st['reward'], done=st['done'], state=st['state'])


_DIGITS = tuple(range(10))
_BCD = (0x00, 0x01, 0x09, 0x10, 0x25, 0x50, 0x99)
# Per game: its reward10 id, its key set's entries per env (0: none), and the RAM bytes its reader reads with what
# they hold in play: a value drawn from a tuple now and then, or a walk [lo, hi] in steps up to the last number.
TRACKED = {
    'smb': (0, 0, {}),                     # from the SMB trajectories
    'pacman': (1, 0, {0x3F: (4, 6, 12, 8, 10, 3), 0x48: (0, 0, 0, 1), 0x47: (0, 0, 0, 1), 0x4A: (0, 0, 1),
                      0x6A: [0, 200, 6], 0x68: (0, 1, 2, 3), 0x67: (3, 2, 1, 0),
                      **{0x70 + i: _DIGITS for i in range(6)}}),
    'contra': (3, 0, {0x18: (5, 5, 5, 4), 0x1C: (0, 0, 1), 0x2C: (4, 4, 3), 0x38: (0, 0, 0, 1), 0x32: (3, 2, 1, 0),
                      0x30: (0, 0, 1, 2, 3), 0x64: [0, 10, 1], 0x65: [0, 255, 12], 0x40: (0, 0, 1),
                      **{0x528 + i: (0, 0, 0x14, 0x11, 5) for i in range(16)},
                      **{0x578 + i: [0, 40, 3] for i in range(16)},
                      0x25: (0, 0, 1), 0x90: (1, 1, 1, 2, 0), 0x7E2: [0, 255, 5], 0x7E3: (0, 0, 1)}),
    'castlevania': (4, 4096, {0x18: (5, 5, 5, 6, 7, 13), 0x19: (6, 6, 6, 5), 0x45: [0, 64, 4],
                              0x28: (0, 0, 1, 2, 3, 6), 0x41: [0, 7, 1], 0x40: [0, 255, 16], 0x3F: [0, 255, 24],
                              0x1A9: [0, 70, 6], 0x22: (0, 0, 1), 0x46C: (0, 0, 8), 0x2A: (3, 2, 1), 0x7FC: _BCD,
                              0x7FD: _BCD, 0x7FE: _BCD}),
    'gradius': (5, 0, {0x00: (5, 5, 5, 4), 0x0A: (1, 1, 0), 0x1B: (0x80, 0x81, 0x80, 0xA0, 0xA1, 192, 0x40),
                       0x20: (3, 2, 1, 0, 255), 0x15: (0, 0, 1), 0x19: (0, 0, 1, 2, 3), 0x3F: [0, 30, 1],
                       0x3E: [0, 255, 12], 0x7E4: _BCD, 0x7E5: _BCD, 0x7E6: _BCD}),
}


def _recorded_ram(case, seed):
    """u8 [T, N, 2048]: each step every listed byte keeps its value with p 0.8, else draws or walks; the rest of the
    RAM holds what it held."""
    n, t = case['envs'], case['steps']
    if case['game'] == 'smb':
        packed = torch.from_numpy(synth.smb_ram15(seed, n, t)).to(DEVICE)
        ram = torch.zeros(t, n, 2048, dtype=torch.uint8, device=DEVICE)
        ram[:, :, list(synth.SMB_ADDRS)] = packed[:, :, :15]
        return ram
    spec = TRACKED[case['game']][2]
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    ram = torch.randint(0, 256, (n, 2048), generator=gen, device=DEVICE, dtype=torch.uint8).expand(t, n, 2048)
    ram = ram.contiguous()
    for a, c in spec.items():
        keep = torch.rand(t, n, generator=gen, device=DEVICE) < 0.8
        if isinstance(c, tuple):
            drawn = torch.tensor(c, device=DEVICE)[torch.randint(0, len(c), (t, n), generator=gen, device=DEVICE)]
            keep[0] = False
            drawn[0] = c[0]
            at = torch.arange(t, device=DEVICE)[:, None].where(~keep, torch.zeros((), dtype=torch.long, device=DEVICE))
            value = drawn.gather(0, at.cummax(0).values)
        else:
            lo, hi, most = c
            step = torch.randint(-most, most + 1, (t, n), generator=gen, device=DEVICE) * ~keep
            at = torch.randint(lo, hi + 1, (n,), generator=gen, device=DEVICE) + step.cumsum(0) - lo
            span = max(hi - lo, 1)       # a walk folded back at its ends
            value = lo + (span - (at.remainder(2 * span) - span).abs())
        ram[:, :, a] = value.to(torch.uint8)
    return ram


def _frames(n, t, seed):
    """Emulated frames of each env-step: 4 a decision, more over a restart, 1 when stepped by the frame."""
    gen = torch.Generator(device=DEVICE).manual_seed(seed + 1)
    pick = torch.tensor([4, 4, 4, 8, 1], dtype=torch.int32, device=DEVICE)
    return pick[torch.randint(0, 5, (t, n), generator=gen, device=DEVICE)]


def _prepare_tracker(case, seed):
    n, t = case['envs'], case['steps']
    gid, cap, _ = TRACKED[case['game']]
    new = lambda *shape, dtype=torch.uint8: torch.zeros(shape, dtype=dtype, device=DEVICE)  # noqa: E731
    return dict(lib=bind_library(hip_library()), gid=gid, n=n, t=t, ram=_recorded_ram(case, seed),
                frames=_frames(n, t, seed),
                state=new(n, 80), reader=new(n, 120), keys=new(n * cap + 1, dtype=torch.int32),
                reward=new(t, n, dtype=torch.float64), done=new(t, n), events=new(t, n, dtype=torch.int32),
                level=new(t, n, dtype=torch.int32), deaths=new(t, n, dtype=torch.int32), end=new(t, n))


def _run_tracker(st):
    for k in ('state', 'reader', 'keys'):        # every replay starts from fresh envs
        st[k].zero_()
    _ok(st['lib'], st['lib'].rl10_run(st['gid'], _ptr(st['ram']), st['t'], st['n'], _ptr(st['frames']), _ptr(st['state']),
                                      _ptr(st['reader']), _ptr(st['keys']), _ptr(st['reward']), _ptr(st['done']),
                                      _ptr(st['events']), _ptr(st['level']), _ptr(st['deaths']), _ptr(st['end']),
                                      _stream()))
    return {k: st[k] for k in ('reward', 'done', 'events', 'level', 'deaths', 'end', 'state')}


# ------------------------------------------------------------------------------------------------ the interface

_PREPARE = dict(env=_prepare_env, rollout=_prepare_rollout, minibatch=_prepare_minibatch, smb=_prepare_smb,
                tracker=_prepare_tracker)
_RUN = dict(env=_run_env, rollout=_run_rollout, minibatch=_run_minibatch, smb=_run_smb, tracker=_run_tracker)


def prepare(case, seed):
    return case['kind'], _PREPARE[case['kind']](case, seed)


def run(state):
    return _RUN[state[0]](state[1])


# One decision of one console: action in; 4 pictures with their emphasis, pads, masks, timeline and the scalars out.
_DECISION = 2 + FRAME_BYTES + 4 * 224 + 4 + 19 + 8 * 45 + 4 + 1 + 4 + 28


def work(case):
    kind, n = case['kind'], case['envs']
    if kind == 'env':
        n *= len(case['boards'].split(','))
        return dict(bytes=n * (_DECISION + (PACKED_BYTES if case['pack6'] else 0)), flops=0)
    if kind == 'rollout':
        return dict(bytes=n * (_DECISION - FRAME_BYTES + PACKED_BYTES), flops=0)
    if kind == 'minibatch':
        return dict(bytes=2 * case['batch'] * case['rows'] * (PACKED_BYTES + FRAME_BYTES), flops=0)
    steps = n * case['steps']
    if kind == 'smb':
        return dict(bytes=steps * (15 + 4 + 1) + 160 * n, flops=0)
    read = len(TRACKED[case['game']][2]) or 15
    return dict(bytes=steps * (read + 4 + 8 + 1 + 4 + 4 + 4 + 1) + 400 * n, flops=0)


def tolerance(case):
    """Every output is defined bit for bit: pictures, hashes and flags are whole numbers, and the rewards are doubles
    added in a stated order (and, where they come as float32, rounded once)."""
    return 'exact'


# ------------------------------------------------------------------------------------------------ 64-bit reference


def exact(case, seed):
    """The SMB tracker's rewards and done flags in float64. The other kinds' results are an emulated machine's (or
    whole numbers throughout), which no closed computation gives."""
    n, t = case['envs'], case.get('steps')
    if case['kind'] == 'tracker' and case['game'] == 'smb':
        reward, done = _smb_reward(synth.smb_ram15(seed, n, t).astype(np.int64), _frames(n, t, seed).cpu().numpy())
        return dict(reward=torch.from_numpy(reward), done=torch.from_numpy(done.astype(np.uint8)), events=None,
                    level=None, deaths=None, end=None, state=None)
    if case['kind'] != 'smb':
        return None
    reward, done = _smb_reward(synth.smb_ram15(seed, n, t).astype(np.int64), np.full((t, n), 4))
    return dict(reward=torch.from_numpy(reward), done=torch.from_numpy(done.astype(np.uint8)), state=None)


# SMB's constants: progress unit, score unit, stall limit in frames, idle penalty a frame.
_SMB = (3000.0, 200.0, 7200, -0.00025)


def _smb_reward(b, frames):
    """RewardTracker.update over [T, N] env-steps, all envs of a step at once. b: the 15 bytes of each;
    frames: the emulated frames of each."""
    t_all, n, _ = b.shape
    signed = lambda v: (v ^ 0x80) - 0x80  # noqa: E731
    mode, routine = b[..., 7], b[..., 0]
    in_play = (mode == 1) & (b[..., 8] == 3)
    level = b[..., 6] * 4 + b[..., 5]
    progress = (signed(b[..., 1]) * 256 + b[..., 2]).astype(np.float64)
    valid = in_play & (routine == 8)
    dying = (mode == 1) & ((routine == 6) | (routine == 11) | ((routine == 8) & (b[..., 3] >= 2)))
    score = sum(b[..., 9 + i] * 10 ** (6 - i) for i in range(6)).astype(np.float64)
    over, won = mode == 3, (mode == 2) & (b[..., 6] == 7)
    reward, dones = np.zeros((t_all, n)), np.zeros((t_all, n), bool)
    best_level, best = np.full(n, -1), np.zeros(n)
    has_best, done = np.zeros(n, bool), np.zeros(n, bool)
    used, idle = np.zeros(n), np.zeros(n, np.int64)
    unit, score_unit, stall, idle_rate = _SMB
    for t in range(t_all):
        live = ~done
        r = np.zeros(n)
        first = live & in_play[t] & (best_level < 0)
        skip = live & in_play[t] & (best_level >= 0) & (level[t] > best_level + 1)
        up = live & in_play[t] & (best_level >= 0) & (level[t] == best_level + 1)
        r += np.where(up, 1.0, 0.0)
        best_level = np.where(first | up, level[t], best_level)
        has_best &= ~(first | up)
        used = np.where(first | up, 0.0, used)
        here = live & in_play[t] & (level[t] == best_level) & valid[t]
        gain = here & has_best & (progress[t] > best)
        r += np.where(gain, (progress[t] - best) / unit, 0.0)
        best = np.where(gain | (here & ~has_best), progress[t], best)
        has_best |= here
        fresh = up | gain
        if t > 0:
            both = in_play[t] & in_play[t - 1]
            lost = dying[t] & ~dying[t - 1]
            death = live & lost & (in_play[t] | in_play[t - 1])
            r += np.where(death, -0.1, 0.0)
            fresh |= death
            some = np.minimum(np.minimum(0.02 * (score[t] - score[t - 1]) / score_unit, 0.1), 0.2 - used)
            pays = live & both & (score[t] > score[t - 1]) & (some > 0)
            r += np.where(pays, some, 0.0)
            used = np.where(pays, used + some, used)
            seen = both & valid[t] & valid[t - 1]
            back = live & ~skip & ~lost & ~dying[t] & ~dying[t - 1] & ~won[t] & ~over[t] & seen & \
                (level[t] == level[t - 1]) & (level[t] == best_level) & (progress[t - 1] - progress[t] >= 0.25 * unit)
            r += np.where(back, -0.02, 0.0)
            r += np.where(live & ~skip & ~fresh & seen & (progress[t] <= progress[t - 1]), idle_rate * frames[t], 0.0)
        idle = np.where(live, 0 if t == 0 else np.where(fresh, 0, idle + frames[t]), idle)
        win = live & won[t]
        r += np.where(win, 5.0, 0.0)
        lose = live & ~won[t] & over[t]
        stalled = live & ~win & ~lose & ~skip & (idle >= stall)
        r += np.where(stalled, -0.1, 0.0)
        done |= skip | win | lose | stalled
        reward[t], dones[t] = r, done
    return reward, dones
