// The reward10 SMB tracker on its own (rl10_smb_run) over T x N env-steps, in one kernel (rlenv_hip.hip k_smb_run).
//
// RewardTracker.update (rl/csrc/reward10.cuh:546-632, env_dev.h ev::update) carries a small state from step to step;
// one env's steps are a chain, and its length times the time of a step is what a call takes (8192 envs are 128 waves
// for 1024 SIMDs: nothing hides a step's latency). So the chain is cut down to the state, and the state in two that
// run one behind the other on waves of their own, kSmbEnvs envs a workgroup, kSmbSteps steps at a time through LDS:
//
// 1. smb_step, every env-step on its own (the workgroup's other waves): the SMB signals of steps t - 1 and t
//    (rl/csrc/reward10.cuh:143-158; the tracker's saved ones before the first step) and all that depends only on them.
// 2. SmbLevels::step, one env per lane: the best level and the best progress (about 30 instructions).
// 3. SmbBudget::step, one env per lane: the score budget, the idle frames and the end (about 30 instructions).
//    Neither chain looks at whether the tracker is done: the third keeps the state as the ending step left it.
// 4. smb_reward, every env-step on its own: the reward, summed in update's order from those terms (so the same
//    doubles are added in the same order: bit-exact), and the done flag.
#pragma once
#include "env_dev.h"

namespace ev {

constexpr int kSmbEnvs = 32, kSmbSteps = 24, kSmbHelpers = 6;   // helpers: the waves of passes 1 and 4, 2 steps a lane
static_assert(kSmbHelpers * 64 * 2 == kSmbEnvs * kSmbSteps, "two steps of one env per helper lane");

// A step's flags: from its signals, then (DC_) as the level chain saw it.
enum : uint32_t {
    ST_IN_PLAY = 1, ST_VALID = 2, ST_WON = 4, ST_OVER = 8, ST_DEATH = 16, ST_DYING = 32, ST_ROLLBACK = 64,
    ST_IDLE = 128, ST_FIRST = 256,
    DC_LEVEL = 1u << 9, DC_GAIN = 1u << 10, DC_SKIP = 1u << 11, DC_AT_BEST = 1u << 12, DC_BETTER = 1u << 13,
    DC_RESET = 1u << 14
};
// Sentinels that keep the chains free of flags. kSmbNoBest: below every progress (so "progress > best" also covers the
// first setting); kSmbNoLevel: a best level not yet seen, above every level; kSmbNotInPlay: a level below every other.
constexpr int32_t kSmbNoBest = (int32_t)0x80000000u, kSmbNoLevel = 0x40000000, kSmbNotInPlay = -0x10000000;

// The SMB signals (env_dev.h smb_signals) of one env-step's 16 packed bytes.
struct SmbSignals {
    uint32_t flags;                    // ST_IN_PLAY, ST_VALID, ST_WON, ST_OVER, ST_DYING
    int32_t level, progress, score;    // (a score of six bytes as digits is below 2^29)
};
__device__ __forceinline__ SmbSignals smb_step_signals(const uint4& q) {
    auto byte = [](uint32_t w, int i) { return (w >> (8 * i)) & 0xFFu; };
    const uint32_t routine = byte(q.x, 0), world = byte(q.y, 2), mode = byte(q.y, 3);
    const bool in_play = mode == 1u && byte(q.z, 0) == 3u;
    SmbSignals s;
    s.flags = (in_play ? ST_IN_PLAY : 0u) | (in_play && routine == 8u ? ST_VALID : 0u) |
              (mode == 2u && world == 7u ? ST_WON : 0u) | (mode == 3u ? ST_OVER : 0u) |
              (mode == 1u && (routine == 6u || routine == 11u || (routine == 8u && byte(q.x, 3) >= 2u)) ? ST_DYING : 0u);
    s.level = (int32_t)(world * 4u + byte(q.y, 1));
    s.progress = (int32_t)(int8_t)byte(q.x, 1) * 256 + (int32_t)byte(q.x, 2);
    uint32_t sc = byte(q.z, 1);
    sc = sc * 10u + byte(q.z, 2);
    sc = sc * 10u + byte(q.z, 3);
    sc = sc * 10u + byte(q.w, 0);
    sc = sc * 10u + byte(q.w, 1);
    sc = sc * 10u + byte(q.w, 2);
    s.score = (int32_t)(sc * 10u);
    return s;
}
// The same from the tracker's saved signals of the step before the first.
__device__ __forceinline__ SmbSignals smb_saved_signals(const Rl10Signals& p) {
    SmbSignals s;
    s.flags = (p.in_play ? ST_IN_PLAY : 0u) | (p.progress_valid ? ST_VALID : 0u) | (p.won ? ST_WON : 0u) |
              (p.game_over ? ST_OVER : 0u) | (p.dying ? ST_DYING : 0u);
    s.level = p.level;
    s.progress = (int32_t)p.progress;
    s.score = !p.has_score || p.score > 0x7FFFFFFF ? 0x7FFFFFFF : (int32_t)p.score;   // (no score: nothing is above it)
    return s;
}

// Pass 1 for one env-step: signals s, the previous step's p (had: there was one). .x the level (kSmbNotInPlay out of
// play), .y the progress (kSmbNoBest where it is not valid), .z the flags; the capped score reward apart (0: none).
__device__ __forceinline__ uint4 smb_step(const SmbSignals& s, const SmbSignals& p, bool had, const Rl10Game& G,
                                          double* score) {
    const uint32_t both = had ? s.flags & p.flags : 0u, any = s.flags | p.flags;
    uint32_t f = (s.flags & (ST_IN_PLAY | ST_VALID | ST_WON | ST_OVER)) | (had ? 0u : ST_FIRST);
    // update's death, before its in-play test (the rollback condition uses it as is)
    const bool death = had && (s.flags & ST_DYING) && !(p.flags & ST_DYING);
    if (death && (any & ST_IN_PLAY)) f |= ST_DEATH;
    double sr = 0.0;
    if ((both & ST_IN_PLAY) && s.score > p.score) {
        sr = kWScore * (double)(s.score - p.score) / G.score_unit;
        if (kScoreCap < sr) sr = kScoreCap;
    }
    *score = sr;
    const bool seen = (both & (ST_IN_PLAY | ST_VALID)) == (ST_IN_PLAY | ST_VALID);
    if (seen && !(any & ST_DYING) && !(s.flags & (ST_WON | ST_OVER)) && s.level == p.level &&
        (double)(p.progress - s.progress) >= kRollbackDrop * G.progress_unit)
        f |= ST_ROLLBACK;
    if (seen && s.progress <= p.progress) f |= ST_IDLE;
    return uint4{(uint32_t)((s.flags & ST_IN_PLAY) ? s.level : kSmbNotInPlay),
                 (uint32_t)((s.flags & ST_VALID) ? s.progress : kSmbNoBest), f, 0u};
}

// Pass 2: update's level and progress logic. update leaves best_progress as it was when a new level clears
// has_best_progress, so the value last assigned is kept apart (last, kSmbNoBest: none in this run) for the state written
// back. step returns what the later passes need: .x the best level after the step, .y the best progress before it
// (after a new level's reset), .z last, .w the flags.
struct SmbLevels {
    int32_t level, best, last;
    __device__ __forceinline__ uint4 step(const uint4& q) {
        const int32_t at = (int32_t)q.x, progress = (int32_t)q.y;
        // (the next step waits for level and best only: a compare and a select, a select and a maximum)
        const bool up = at - 1 == level, skip = at - 1 > level;
        const bool first = level == kSmbNoLevel && at >= 0;          // in play and no best level yet
        const bool reset = up || first;
        level = reset ? at : level;
        const int32_t before = reset ? kSmbNoBest : best;
        const bool at_best = at == level;
        const int32_t reached = at_best ? progress : kSmbNoBest;
        const bool better = reached > before;                        // a first setting or a gain
        const bool gain = better && before != kSmbNoBest;
        best = reached > before ? reached : before;
        last = better ? progress : last;
        const uint32_t f = q.z | (up ? DC_LEVEL : 0u) | (gain ? DC_GAIN : 0u) | (skip ? DC_SKIP : 0u) |
                           (at_best ? DC_AT_BEST : 0u) | (better ? DC_BETTER : 0u) | (reset ? DC_RESET : 0u);
        return uint4{(uint32_t)level, (uint32_t)before, (uint32_t)last, f};
    }
};

// Pass 3: update's score budget, idle frames, deaths and end. step takes the flags as the level chain left them, returns
// whether the step would end the episode, and puts the score term (<= 0: none) over the capped score reward. The budget
// is spent by max(term, 0): adding +0.0 leaves it as it is.
struct SmbBudget {
    double used;
    int64_t idle;
    int32_t deaths;
    __device__ __forceinline__ bool step(uint32_t f, double* score, int frames, int64_t stall) {
        used = (f & DC_RESET) ? 0.0 : used;
        const double sr = __builtin_fmin(kScoreBudget - used, *score);   // (both finite)
        used += __builtin_fmax(sr, 0.0);
        *score = sr;
        deaths += (int32_t)((f >> 4) & 1u);   // ST_DEATH
        const int64_t more = idle + frames;
        idle = (f & (DC_LEVEL | DC_GAIN | ST_DEATH | ST_FIRST)) ? 0 : more;
        return (f & (DC_SKIP | ST_WON | ST_OVER)) || idle >= stall;
    }
};

// update's end reason from the flags of the step that ended the episode (checked in update's order): 2 won, 1 game
// over, 3 skipped a level, else 4 stalled.
__device__ __forceinline__ uint32_t smb_end_reason(uint32_t f) {
    return (f & ST_WON) ? 2u : (f & ST_OVER) ? 1u : (f & DC_SKIP) ? 3u : 4u;
}

// Pass 4 for one env-step that the tracker took: update's reward, its terms added in update's order. d: pass 2's
// record, score: pass 3's term, ends: the step ended the episode.
__device__ __forceinline__ double smb_reward(const uint4& d, double score, bool ends, int frames, const Rl10Game& G) {
    const uint32_t f = d.w;
    const bool death = (f & ST_DEATH) != 0, skip = (f & DC_SKIP) != 0;
    const bool fresh = (f & (DC_LEVEL | DC_GAIN)) != 0 || death;
    double r = 0.0;
    if (f & DC_LEVEL) r += kWLevel;
    if (f & DC_GAIN) r += kWProgress * ((double)(int32_t)d.z - (double)(int32_t)d.y) / G.progress_unit;
    if (death) r += kWDeath;
    if (score > 0.0) r += score;
    if ((f & ST_ROLLBACK) && !skip && (f & DC_AT_BEST)) r += kWRollback;
    if (!fresh && !skip && (f & ST_IDLE)) r += G.idle_per_frame * frames;
    if (f & ST_WON) r += kWWin;
    else if (ends && !(f & (ST_OVER | DC_SKIP))) r += kWStall;
    return r;
}

}  // namespace ev
