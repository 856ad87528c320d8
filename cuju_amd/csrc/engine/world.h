// SPDX-License-Identifier: Apache-2.0
// Restates game logic of cuju (Copyright 2026 The cuju Authors), a reimplementation of Google
// Research Football (Copyright 2019 Google LLC); see NOTICE.
// World access, frame mirroring, the world RNG and the per-player helpers every stage reads.
// Semantics: include/cuju/simulation/world.h:37-167 (frames and mirrors),
// include/cuju/simulation/access.h:13-63, include/cuju/simulation/humanoid.h:118-420,
// include/cuju/rng.h:18-113 (Boost MT19937 + uniform_real in the world's 2512 RNG bytes).
#pragma once

#include "tables.h"

namespace eng {

// ---- faults ----------------------------------------------------------------------------------------
// A path GRF leaves undefined. `Fail` returns false for the caller to propagate; `Fatal` marks a
// state no match reaches (list overflow, a team without players).
#if defined(__HIPCC__)
// 1 = a path GRF leaves undefined, 2 = a state no match reaches; the batch reads it after a launch.
// Each device build (one per group width) holds its own.
static __device__ uint32_t gEngineFault;
#endif
#if !ENG_DEVICE
const char *&FailReason();
[[noreturn]] void FatalHost(const char *message);
// The ticks this host thread has run, for the host build's per-step tick counts.
inline long long &HostTicks() {
    static thread_local long long ticks = 0;
    return ticks;
}
#endif
HD void Unsupported(const char *reason) {
#if ENG_DEVICE
    (void)reason;
    gEngineFault = 1;
#else
    FailReason() = reason;
#endif
}
HD void Fatal(const char *reason) {
#if ENG_DEVICE
    (void)reason;
    gEngineFault = 2;
#else
    FatalHost(reason);
#endif
}
HD bool Fail(const char *reason) {
    Unsupported(reason);
    return false;
}

using PlayerList = Small<int, kPlayers>;

// ---- the world's random numbers --------------------------------------------------------------------
// Boost.Random's mt19937 drawn through uniform_real<float>, over the world's RNG bytes: the 624
// state words, then the index of the next word (8 bytes at 2496) and the distribution's bounds
// (floats at 2504 and 2508).
struct Rng {
    static constexpr int kWords = 624, kShift = 397, kIndexAt = 2496, kLowAt = 2504, kHighAt = 2508;
    static constexpr uint32_t kTop = 0x80000000u, kTwist = 0x9908b0dfu;
    GlobalPointer<uint8_t> b;
    template <class T>
    HD T Load(int at) const {
        T v;
        memcpy(&v, b + at, sizeof v);
        return v;
    }
    template <class T>
    HD void Store(int at, T v) {
        memcpy(b + at, &v, sizeof v);
    }
    HD uint32_t Word(int i) const { return Load<uint32_t>(4 * i); }
    // Word `i` of the next generation, from its top bit, the following word's low bits and the word
    // kShift ahead, indices wrapping; the words are renewed in order, so the wrapped ones read
    // are already new.
    HD uint32_t Renewed(int i) const {
        const uint32_t next = Word((i + 1) % kWords);
        const uint32_t joined = (Word(i) & kTop) | (next & ~kTop);
        return Word((i + kShift) % kWords) ^ (joined >> 1) ^ ((next & 1) * kTwist);
    }
    // Knuth's multiplier fills the words from the seed. Boost then sets the first word's low bits as
    // a generation step would, from words 396 and 623, and turns an all-zero state into a lone top
    // bit.
    HDN void Seed(uint32_t seed) {
        uint32_t word = seed;
        Store(0, word);
        for (int i = 1; i < kWords; i++) {
            word = 1812433253u * (word ^ (word >> 30)) + (uint32_t)i;
            Store(4 * i, word);
        }
        Store<uint64_t>(kIndexAt, kWords);
        uint32_t y = Word(kShift - 1) ^ Word(kWords - 1);
        y = (y & kTop) ? (((y ^ kTwist) << 1) | 1) : (y << 1);
        Store(0, (Word(0) & kTop) | (y & ~kTop));
        bool zero = true;
        for (int i = 0; i < kWords && zero; i++) zero = Word(i) == 0;
        if (zero) Store(0, kTop);
    }
    HDN void Generate() {
        for (int i = 0; i < kWords; i++) Store(4 * i, Renewed(i));
        Store<uint64_t>(kIndexAt, 0);
    }
    // The next word, tempered.
    HD uint32_t Next() {
        if (Load<uint64_t>(kIndexAt) == kWords) Generate();
        const uint64_t i = Load<uint64_t>(kIndexAt);
        Store<uint64_t>(kIndexAt, i + 1);
        uint32_t y = Word((int)i);
        y ^= y >> 11;
        y ^= (y << 7) & 0x9d2c5680u;
        y ^= (y << 15) & 0xefc60000u;
        return y ^ (y >> 18);
    }
    // A float in [low, high): the word over 2^32 in float, scaled and moved; a draw that rounds up
    // to `high` is drawn again.
    HD float Uniform() {
        const float low = Load<float>(kLowAt), high = Load<float>(kHighAt);
        for (;;) {
            const float r = (float)Next() / 4294967296.0f * (high - low) + low;
            if (r < high) return r;
        }
    }
};
HD float RandomInRange(World &w, float lo, float hi) {
    Rng g{w.rng};
    float stretch = hi - lo;
    return lo + (g.Uniform() * stretch);
}

// ---- mirroring between team frames ----------------------------------------------------------------
HD void MirrorRadian(Radian &r) { r.rotated = !r.rotated; }

HDN void MirrorHumanoid(GlobalRef<Humanoid> humanoid, bool &mirrored) {
    Humanoid &h = humanoid;
    NodeState &root = h.nodes[0];
    root.position = root.position * Vec3(-1, -1, 1);
    Quat q = root.rotation;
    root.rotation = mirrored ? Quat(q.q[1], q.q[0], -q.q[3], q.q[2]) : Quat(q.q[1], q.q[0], q.q[3], -q.q[2]);
    mirrored = !mirrored;
    h.startPos.Mirror();
    MirrorRadian(h.startAngle);
    h.nextStartPos.Mirror();
    MirrorRadian(h.nextStartAngle);
    SpatialState &s = h.spatial;
    s.position.Mirror();
    s.actualMovement.Mirror();
    s.physicsMovement.Mirror();
    s.animationMovement.Mirror();
    s.movement.Mirror();
    s.actionSmuggleMovement.Mirror();
    s.movementSmuggleMovement.Mirror();
    s.positionOffsetMovement.Mirror();
    h.prevPosition2D.Mirror();
    h.tripDirection.Mirror();
    h.decayingPositionOffset.Mirror();
}

// The first-processed team's players come first in the player array, the other team's after them.
HD int FirstTeamSize(const World &w) {
    return w.FirstTeamID() == 0 ? w.scenario.leftTeamSize : w.scenario.rightTeamSize;
}
// Mirrors the humanoids of the flagged teams (by team ID). Their players form one range of the
// player array, and each humanoid mirrors on its own, so the lanes of the match take the range's
// players in turn; the caller synchronizes the group before the mirrored state is read.
HD void MirrorTeams(World &w, bool t0, bool t1) {
    for (int t = 0; t < 2; t++)
        if (t == 0 ? t0 : t1) {
            w.flags.teamSide[t] *= -1;
            w.flags.teamMirrored[t] = !w.flags.teamMirrored[t];
        }
    const bool firstFlagged = w.FirstTeamID() == 0 ? t0 : t1, secondFlagged = w.FirstTeamID() == 0 ? t1 : t0;
    const int split = FirstTeamSize(w);
    const int lo = firstFlagged ? 0 : split, hi = secondFlagged ? w.match.playerCount : split;
    for (int p = lo + GroupRank(); p < hi; p += kGroupLanes)
        MirrorHumanoid(w.match.players[p].base.humanoid, w.flags.humanoidMirrored[p]);
}

// Prediction and history arrays mirror lazily: `lazyFlip` says they hold negated x and y.
HD void MirrorBall(Ball &b) {
    b.momentum.Mirror();
    b.lazyFlip = !b.lazyFlip;
    b.positionBuffer.Mirror();
}
// Negates x and y of `count` stored vectors; the lanes of the match take four entries each per
// round, so their reads overlap in flight. Every lane of the match calls it.
HD void MirrorStored(Vec3 *a, int count) {
    constexpr int kRun = 4;
    for (int base = GroupRank() * kRun; base < count; base += kRun * kGroupLanes) {
        Vec3 v[kRun];
        for (int j = 0; j < kRun; j++)
            if (base + j < count) v[j] = a[base + j];
        for (int j = 0; j < kRun; j++)
            if (base + j < count) {
                v[j].Mirror();
                a[base + j] = v[j];
            }
    }
}
HD void BallMaterialize(Ball &b) {
    if (!b.lazyFlip) return;
    MirrorStored(b.predictions, 401);
    MirrorStored(b.positionHistory.e, b.positionHistory.count);
    GroupSync();
    b.lazyFlip = false;
}
// Entry `i` (below the count) of a mental image's players, its team's lazy mirror applied.
HD PlayerImage MentalImageEntry(const World &w, const MentalImage &m, int i) {
    PlayerImage p = m.players[i];
    if (m.lazyTeamFlip[w.playerTeamID[p.player]]) {
        p.position.Mirror();
        p.directionVector.Mirror();
        p.movement.Mirror();
    }
    return p;
}
// Applies an image's lazy mirrors to its stored predictions and player images.
HD void MentalMaterialize(const World &w, MentalImage &m) {
    if (m.lazyFlip)
        for (int i = 0; i < m.ballPredictions.count; i++) m.ballPredictions[i].Mirror();
    m.lazyFlip = false;
    for (int i = 0; i < m.players.count; i++) m.players[i] = MentalImageEntry(w, m, i);
    m.lazyTeamFlip[0] = m.lazyTeamFlip[1] = false;
}

// Player images mirror lazily per team, the ball's predictions lazily as a whole.
HD void MirrorMentalImage(World &w, int k, bool t0, bool t1, bool ball) {
    MentalImage &m = w.match.mentalImages[k];
    m.lazyTeamFlip[0] ^= t0;
    m.lazyTeamFlip[1] ^= t1;
    if (ball) {
        m.lazyFlip = !m.lazyFlip;
        w.flags.mentalBallMirrored[k] = !w.flags.mentalBallMirrored[k];
    }
}

HDN void MirrorMatch(GlobalRef<World> world, bool t0, bool t1, bool ball) {
    World &w = world;
    ENG_SCOPE(18);
    if (!t0 && !t1 && !ball) {
        GroupSync();
        return;
    }
    MirrorTeams(w, t0, t1);
    if (ball) {
        w.flags.ballMirrored = !w.flags.ballMirrored;
        MirrorBall(w.match.ball);
    }
    for (int k = 0; k < w.match.mentalImages.count; k++) MirrorMentalImage(w, k, t0, t1, ball);
    GroupSync();
}

// A state stores the ball, last-touch team IDs and referee team/positions in canonical order; the
// conversion is an involution.
HDN void CanonicalToRest(GlobalRef<World> world) {
    World &w = world;
    MatchState &m = w.match;
    if (w.FirstTeamID() == 1) {
        for (int i = 0; i < 4; i++)
            if (m.lastTouchTeamIDs[i] != -1) m.lastTouchTeamIDs[i] = 1 - m.lastTouchTeamIDs[i];
        if (m.lastTouchTeamID != -1) m.lastTouchTeamID = 1 - m.lastTouchTeamID;
    }
    if (!w.scenario.reverseTeamProcessing) return;
    MirrorBall(m.ball);
    for (int k = 0; k < m.mentalImages.count; k++) m.mentalImages[k].lazyFlip = !m.mentalImages[k].lazyFlip;
    m.referee.buffer.teamID = 1 - m.referee.buffer.teamID;
    m.referee.buffer.restartPos.Mirror();
    m.referee.foul.foulPosition.Mirror();
}
HD void RestToCanonical(World &w) { CanonicalToRest(w); }

// ---- access ---------------------------------------------------------------------------------------
HD int TeamSlot(const World &w, int teamID) { return teamID == w.FirstTeamID() ? 0 : 1; }
HD Team &TeamByID(World &w, int teamID) { return w.match.teams[TeamSlot(w, teamID)]; }
HD const Team &TeamByID(const World &w, int teamID) { return w.match.teams[TeamSlot(w, teamID)]; }
HD const Team &TeamOfPlayer(const World &w, int p) { return TeamByID(w, w.playerTeamID[p]); }
HD const Team &OpponentTeamOfPlayer(const World &w, int p) { return TeamByID(w, 1 - w.playerTeamID[p]); }
HD Humanoid &Hum(World &w, int p) { return w.match.players[p].base.humanoid; }
HD const Humanoid &Hum(const World &w, int p) { return w.match.players[p].base.humanoid; }
HD SpatialState &Sp(World &w, int p) { return w.match.players[p].base.humanoid.spatial; }
HD const SpatialState &Sp(const World &w, int p) { return w.match.players[p].base.humanoid.spatial; }

// GRF: the time compares as unsigned, so a negative time reads the entry at 2990 ms.
HD Vec3 BallPredictRaw(const Vec3 *pred, int ms) {
    int i = ms;
    if ((uint32_t)i >= kBallPredictionSpanMs) i = kBallPredictionSpanMs - 10;
    i = i / 10;
    if (i < 0) i = 0;
    return pred[i];
}
HD Vec3 BallPredict(const Ball &b, int ms) {
    Vec3 v = BallPredictRaw(b.predictions, ms);
    if (b.lazyFlip) v.Mirror();
    return v;
}

HD int HumanGamerCount(const Team &t) {
    int n = 0;
    for (int g = 0; g < t.gamers.count; g++)
        if (!t.gamers[g].controller.keyboard.disabled) n++;
    return n;
}
// Gamers count the first team's, then the second's.
HD HumanGamer &GamerByGlobal(World &w, int g) {
    int first = w.match.teams[0].gamers.count;
    return g < first ? w.match.teams[0].gamers[g] : w.match.teams[1].gamers[g - first];
}
HD const HumanGamer &GamerByGlobal(const World &w, int g) {
    int first = w.match.teams[0].gamers.count;
    return g < first ? w.match.teams[0].gamers[g] : w.match.teams[1].gamers[g - first];
}
HD int GlobalGamerIndex(const World &w, int teamID, int gamer) {
    return TeamSlot(w, teamID) == 0 ? gamer : w.match.teams[0].gamers.count + gamer;
}

// The bookkeeping a state omits, from a loaded state: team IDs, formation overrides and the roster.
HD void InitializePlayerTeams(World &w) {
    const int first = w.FirstTeamID(), firstSize = FirstTeamSize(w);
    for (int p = 0; p < w.match.playerCount; p++) w.playerTeamID[p] = p < firstSize ? first : 1 - first;
    for (int p = 0; p < kPlayers; p++) {
        w.formationOverride[p] = 0;
        w.roster.active[p] = p < w.match.playerCount && w.match.players[p].base.isActive;
        w.roster.timeToBallMs[p] = w.match.players[p].timeToBallMs;
    }
}
// Whether the roster holds the fields it copies (a check of the host build).
HD bool RosterMatches(const World &w) {
    for (int p = 0; p < w.match.playerCount; p++)
        if (w.roster.active[p] != w.match.players[p].base.isActive || w.roster.timeToBallMs[p] != w.match.players[p].timeToBallMs)
            return false;
    return true;
}

HD PlayerList TeamAllPlayers(const World &w, int teamID) {
    PlayerList l;
    for (int p = 0; p < w.match.playerCount; p++)
        if (w.playerTeamID[p] == teamID) l.push_back(p);
    return l;
}
// A set of players, a bit each, read as the list of them in state order: by a loop over the set, or by
// index. A list of up to 22 entries lies on the lane's stack, behind a store for every player and a
// load for every use. Measured, ms per step: 4,096 matches of 32 lanes 37.4 -> 36.6, 8,192 of 16 lanes
// 70.2 -> 68.3, 16,384 of 8 lanes 106.5 -> 104.6.
struct PlayerSet {
    uint32_t mask = 0;
    HD int size() const { return PopCount(mask); }
    HD bool empty() const { return mask == 0; }
    // The n-th player: the half that holds its bit, then half of that half.
    HD int operator[](int n) const {
        int at = 0;
#pragma unroll
        for (int half = 16; half > 0; half >>= 1) {
            const int below = PopCount((mask >> at) & ((1u << half) - 1u));
            const bool above = n >= below;
            n -= above ? below : 0;
            at += above ? half : 0;
        }
        return at;
    }
    struct Iterator {
        uint32_t left;
        HD int operator*() const { return LowestBit(left); }
        HD void operator++() { left &= left - 1; }
        HD bool operator!=(const Iterator &o) const { return left != o.left; }
    };
    HD Iterator begin() const { return Iterator{mask}; }
    HD Iterator end() const { return Iterator{0}; }
    HD operator PlayerList() const {
        PlayerList l;
        for (int p : *this) l.e[l.count++] = p;
        return l;
    }
};
static_assert(kPlayers <= 32, "a set of players is a word");
// The active players of a team. The lanes of the match test the players in turn; every lane of the
// match must make the call.
HD PlayerSet TeamActivePlayers(const World &w, int teamID) {
    PlayerSet s;
    const int players = w.match.playerCount;
#pragma unroll
    for (int base = 0; base < kPlayers; base += kGroupLanes) {
        const int p = base + GroupRank(), at = p < kPlayers ? p : 0;
        s.mask |= (uint32_t)GroupBallot((p < players) & (w.playerTeamID[at] == teamID) & w.roster.active[at]) << base;
    }
    return s;
}
HD int TeamDynamicSide(const World &w, int teamID) { return w.flags.teamSide[teamID]; }

// ---- per-player helpers ----------------------------------------------------------------------------
HD int FormationSource(const World &w, int p) {
    int o = w.formationOverride[p];
    return o ? o - 1 : p;
}
HD const StaticFormation &Formation(const World &w, const Ctx &c, int p) {
    return c.sd->formation[FormationSource(w, p)];
}

HD float FixAngle(float a) { return ModulateIntoRange(-PI, PI, a + 0.5f * PI); }

HD float RangeVelocity(float v) {
    float r = kIdleVelocity;
    if (v >= kIdleDribbleSwitch && v < kDribbleWalkSwitch) r = kDribbleVelocity;
    else if (v >= kDribbleWalkSwitch && v < kWalkSprintSwitch) r = kWalkVelocity;
    else if (v >= kWalkSprintSwitch) r = kSprintVelocity;
    return r;
}
HD int VelocityCat(float v) {
    float r = RangeVelocity(v);
    if (r == kIdleVelocity) return kVelIdle;
    if (r == kDribbleVelocity) return kVelDribble;
    if (r == kWalkVelocity) return kVelWalk;
    if (r == kSprintVelocity) return kVelSprint;
    return kVelIdle;
}
HD float VelocityFloat(int cat) {
    switch (cat) {
        case kVelIdle:
            return kIdleVelocity;
        case kVelDribble:
            return kDribbleVelocity;
        case kVelWalk:
            return kWalkVelocity;
        case kVelSprint:
            return kSprintVelocity;
    }
    return 0;
}
// The quantized velocity of a player.
HD float PlayerFloatVelocity(const World &w, int p) { return VelocityFloat(Sp(w, p).velocityCat); }

// `std::min` operand order: a NaN second operand loses.
HD float MinF(float a, float b) { return (b < a) ? b : a; }
// `std::max(a, b)`: `a` wins a tie or a NaN.
HD float MaxF(float a, float b) { return (a < b) ? b : a; }

HD float TeamDifficulty(const World &w, int teamID) {
    return teamID == 0 ? w.scenario.leftDifficulty : w.scenario.rightDifficulty;
}
HD float GetStatistic(const World &w, const Ctx &c, int p, int stat) {
    float m = 0.3f + 0.7f * TeamDifficulty(w, w.playerTeamID[p]);
    m *= 0.7f + 0.3f * w.match.players[p].base.fatigueFactorInverse;
    return c.sd->data[p].stats[stat] * m;
}
HD bool ExternalControllerActive(const World &w, int p) {
    int ec = w.match.players[p].base.externalController;
    if (ec < 0) return false;
    return !GamerByGlobal(w, ec).controller.keyboard.disabled;
}
HD int GetReactionTimeMs(const World &w, const Ctx &c, int p) {
    int r = TruncToInt32(roundf(80.0f - GetStatistic(w, c, p, kStatReaction) * 40.0f));
    if (ExternalControllerActive(w, p)) return r;
    return TruncToInt32((float)r + (1.0f - TeamDifficulty(w, w.playerTeamID[p])) * 100);
}
HD float GetLastTouchBias(const World &w, int p, int decayMs) {
    uint64_t t = w.match.actualTimeMs;
    if (decayMs > 0)
        return 1.0f - Clamp((float)(t - w.match.players[p].base.lastTouchTimeMs) / (float)decayMs, 0.0f, 1.0f);
    return 0.0f;
}
HD float TeamLastTouchBias(const World &w, int teamID, int decayMs) {
    int lt = TeamByID(w, teamID).lastTouchPlayer;
    return lt >= 0 ? GetLastTouchBias(w, lt, decayMs) : 0.0f;
}
// GRF: before the first touch, the team processed first counts as the last to touch.
HD float MatchLastTouchBias(const World &w, int decayMs) {
    int team = w.match.lastTouchTeamID != -1 ? w.match.lastTouchTeamID : w.FirstTeamID();
    return TeamLastTouchBias(w, team, decayMs);
}

HD void OffsetPosition(World &w, int p, const Vec3 &off) {
    Humanoid &h = Hum(w, p);
    h.nextStartPos += off;
    h.startPos += off;
    h.spatial.position += off;
    h.spatial.positionOffsetMovement += off * 100.0f;
    h.decayingPositionOffset += off;
    if (h.decayingPositionOffset.Length() > 0.1f) h.decayingPositionOffset = h.decayingPositionOffset.Normalized() * 0.1f;
    h.anim.positionOffset += off;
}

HD int MentalImageIndex(const World &w, int historyMs) {
    int i = TruncToInt32(round((double)((float)historyMs / 100.0)));
    if (i >= w.match.mentalImages.count) i = w.match.mentalImages.count - 1;
    if (i < 0) i = 0;
    return i;
}
// The offset from the image's stamp wraps as unsigned 32-bit, so one outside the window (a negative
// one included) reads the last prediction.
// The fields one image's predictions read, looked up once for the many times a caller asks.
struct MentalBallView {
    GlobalPointer<const Vec3> image, ball;
    uint64_t now;
    uint32_t stamp;
    float maxDeviation;
    bool imageFlip, ballFlip;
    HD MentalBallView(const World &w, int k) {
        const MentalImage &m = w.match.mentalImages[k];
        image = m.ballPredictions.e;
        ball = w.match.ball.predictions;
        now = w.match.actualTimeMs;
        stamp = m.timeStampMs;
        maxDeviation = m.maxDistanceDeviation;
        imageFlip = m.lazyFlip;
        ballFlip = w.match.ball.lazyFlip;
    }
    HD Vec3 At(int ms) const {
        int i = (int)(uint32_t)((uint64_t)(int64_t)ms + now - (uint64_t)stamp);
        if ((uint32_t)i >= kBallPredictionSpanMs) i = kBallPredictionSpanMs - 10;
        i = i / 10;
        if (i < 0) i = 0;
        Vec3 r = image[i];
        if (imageFlip) r.Mirror();
        Vec3 real = BallPredictRaw(ball, ms);
        if (ballFlip) real.Mirror();
        return r.EnforceMaximumDeviation(real, maxDeviation);
    }
};
HD Vec3 MentalBallPrediction(const World &w, int k, int ms) { return MentalBallView(w, k).At(ms); }

// Exact: float differences whose squares add in double.
HD float GetDistance(const Vec3 &a, const Vec3 &b) {
    float dx = a.v[0] - b.v[0], dy = a.v[1] - b.v[1], dz = a.v[2] - b.v[2];
    if (dx == 0.0f && dy == 0.0f && dz == 0.0f) return 0.0f;
    double x = dx, y = dy, z = dz;
    float l = (float)sqrt(x * x + y * y + z * z);
    if (l < kAboveMillionth) l = 0;
    return l;
}

HD float Curve(float s, float bias = 1.0f) {
    return (libm::sinf((s - 0.5f) * PI) * 0.5f + 0.5f) * bias + s * (1.0f - bias);
}

HD float GetMaximumVelocity(const StaticData &sd, int p) {
    return kSprintVelocity * (0.9f + sd.data[p].velocityStat * 0.1f);
}

}  // namespace eng
