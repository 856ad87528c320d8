// SPDX-License-Identifier: Apache-2.0
// Restates game logic of cuju (Copyright 2026 The cuju Authors), a reimplementation of Google
// Research Football (Copyright 2019 Google LLC); see NOTICE.
// Keyframe poses, skeleton transforms, and the per-tick application of an animation frame to the
// nodes of a humanoid with GRF's smoothing. Semantics: include/cuju/animation/keyframes.h:16-194,
// include/cuju/animation/skeleton.h:98-222, include/cuju/animation/apply.h:16-367,
// include/cuju/simulation/humanoid.h:178-296 (spatial state).
#pragma once

#include "world.h"

namespace eng {

// The pose of a node at `frame` from its keys, which are in frame order. Past the animation's end,
// the last two keys' motion carries on (one key holds; none gives the identity at the origin). At
// or before frame 0, the first key holds. Between, the keys either side of the frame blend: the
// orientation spherically by the frame's share of the gap, the position by each key's closeness
// (both ratios divided in double and rounded to float once); with a key on one side only, that key
// holds. Also run on the host to fill the interpolation table, so that table reads equal it bit
// for bit.
HDN void ComputeInterpolated(GlobalRef<const Anim> animation, GlobalPointer<const KeyFrame> keys, int keyCount, int frame, Quat &ori, Vec3 &pos) {
    const Anim &a = animation;
    if (frame >= a.frameCount) {
        ori = Quat::Identity();
        pos = Vec3(0);
        if (keyCount == 0) return;
        const KeyFrame &last = keys[keyCount - 1];
        ori = last.orientation;
        pos = last.position;
        if (keyCount == 1) return;
        const KeyFrame &before = keys[keyCount - 2];
        const float gap = (float)(last.frame - before.frame);
        const float beyond = 1 + ((1 / gap) * (float)(frame - last.frame));
        ori = before.orientation.Slerp(beyond, last.orientation);
        pos = before.position * (1 - beyond) + last.position * beyond;
        return;
    }
    if (frame <= 0) {
        ori = keys[0].orientation;
        pos = keys[0].position;
        return;
    }
    int after = 0;
    while (after < keyCount && keys[after].frame < frame) after++;
    if (after == 0 || after == keyCount) {
        const KeyFrame &only = keys[after == 0 ? 0 : keyCount - 1];
        ori = only.orientation;
        pos = only.position;
        return;
    }
    const KeyFrame &from = keys[after - 1], &to = keys[after];
    const double gap = (double)(to.frame - from.frame);
    const float sinceFrom = (float)(frame - from.frame), untilTo = (float)(to.frame - frame);
    const float share = (float)((double)(frame - from.frame) / gap);
    ori = from.orientation.Slerp(share, to.orientation);
    pos = from.position * (float)(1 - sinceFrom / gap) + to.position * (float)(1 - untilTo / gap);
}

HD void Interpolated(const Ctx &c, const Anim &a, const NodeAnim &n, int frame, Quat &ori, Vec3 &pos) {
    if (frame < n.interpFrames) {
        const InterpEntry &e = c.T().interp[n.interpFirst + (frame < 0 ? 0 : frame) * n.interpStride];
        ori = e.orientation;
        pos = e.position;
        return;
    }
    ComputeInterpolated(a, c.T().keys + n.keyFirst, n.keyCount, frame, ori, pos);
}

HD void BlendFrames(Quat at, const Vec3 &pAt, const Quat &next, const Vec3 &pNext, float bias, Quat &ori, Vec3 &pos) {
    at.MakeSameNeighborhood(next);
    ori = at.Lerp(bias, next).Normalized();
    pos = pAt * (1.0f - bias) + pNext * bias;
}

HD void InterpolatedZ(const Ctx &c, const Anim &a, const NodeAnim &n, int frame, Quat &ori, Vec3 &pos, float &z) {
    if (frame < n.interpFrames) {
        const InterpEntry &e = c.T().interp[n.interpFirst + (frame < 0 ? 0 : frame) * n.interpStride];
        ori = e.orientation;
        pos = e.position;
        z = e.angleZ;
        return;
    }
    ComputeInterpolated(a, c.T().keys + n.keyFirst, n.keyCount, frame, ori, pos);
    float x, y;
    ori.Angles(x, y, z);
}

// The node of a body part comes from the animation's map (each body part has at most one node, so
// it is the node a scan of the node list finds first).
HD void GetKeyFrameZ(const Ctx &c, const Anim &a, int bodyPart, int frame, Quat &ori, Vec3 &pos, float &z) {
    const int i = a.nodeOfBodyPart[bodyPart];
    if (i >= 0) {
        InterpolatedZ(c, a, c.T().nodes[a.nodeFirst + i], frame, ori, pos, z);
        return;
    }
    float x, y;
    ori.Angles(x, y, z);
}

HD bool GetKeyFrame(const Ctx &c, const Anim &a, int bodyPart, int frame, Quat &ori, Vec3 &pos) {
    const int i = a.nodeOfBodyPart[bodyPart];
    if (i < 0) return false;
    const NodeAnim &n = c.T().nodes[a.nodeFirst + i];
    Interpolated(c, a, n, frame, ori, pos);
    for (int k = 0; k < n.keyCount; k++)
        if (c.T().keys[n.keyFirst + k].frame == frame) return true;
    return false;
}

// ---- skeleton transforms -------------------------------------------------------------------------
// A node's transform in the world.
struct Transform {
    Vec3 position, scale;
    Quat rotation;
};
// A local transform placed under `parent`. A relative one composes with it: the rotations
// multiplied and renormalized, the scales multiplied, the position scaled and turned by the
// parent's, then moved by its position. An absolute one, or a root's, stands as it is.
HD Transform Placed(const Transform *parent, int localMode, const Vec3 &pos, const Quat &rot, const Vec3 &scale) {
    if (localMode != kLocalRelative || !parent) return Transform{pos, scale, rot};
    Transform t;
    t.rotation = (parent->rotation * rot).Normalized();
    t.scale = parent->scale * scale;
    t.position = parent->rotation * (parent->scale * pos) + parent->position;
    return t;
}
// Every node's world transform, parents before children (the skeleton lists them so).
HD void WorldTransforms(const Skeleton &sk, const NodeState *nodes, Transform *out) {
    for (int n = 0; n < sk.nodeCount; n++) {
        const int up = sk.nodes[n].parent;
        out[n] = Placed(up >= 0 ? &out[up] : nullptr, nodes[n].localMode, nodes[n].position, nodes[n].rotation, nodes[n].scale);
    }
}

// A mesh's box in the world: placed under its node, turned by the placed rotation and moved to
// the placed position (GRF leaves the scale out of the box).
HD WorldGeometry PlacedGeometry(const SkelGeometry &g, const Transform &node) {
    const Transform at = Placed(&node, g.localMode, g.position, g.rotation, g.scale);
    return WorldGeometry{Aabb{g.boxMin, g.boxMax}.Rotated(at.rotation).Translated(at.position), at.position};
}

// One of a node's geometries in the world: the transforms down from the root to the node (the path
// packed root first, four bits a node), then the geometry's.
static_assert(kHumanoidNodes <= 15, "a node's index and one to spare fit four bits");
HDN WorldGeometry PlacedPart(GlobalRef<const Skeleton> skeleton, GlobalPointer<const NodeState> nodes, int node, int geometry) {
    const Skeleton &sk = skeleton;
    uint64_t path = 0;
    for (int n = node, up; n >= 0; n = up < n ? up : -1) {
        path = path << 4 | (uint64_t)(n + 1);
        up = sk.nodes[n].parent;  // parents come before their children
    }
    Transform at;
    const Transform *parent = nullptr;
    for (; path; path >>= 4) {
        const NodeState &s = nodes[(int)(path & 15) - 1];
        at = Placed(parent, s.localMode, s.position, s.rotation, s.scale);
        parent = &at;
    }
    return PlacedGeometry(sk.nodes[node].geometries[geometry], at);
}

// ---- applying a frame ------------------------------------------------------------------------------
HD float SmoothBeginBias(int frame) {
    int f = frame < 0 ? 0 : frame > 8 ? 8 : frame;
    return libm::PowfPos(Curve(1.0f - NormalizedClamp((float)f, 0, 8), 1.0f), 0.5f);
}
HD int JointSpeedClass(int bp) {
    if (bp == kBpLeftElbow || bp == kBpRightElbow || bp == kBpLeftKnee || bp == kBpRightKnee) return 1;
    if (bp == kBpLeftAnkle || bp == kBpRightAnkle) return 2;
    return 0;
}
HD float JointSpeedLimit(int cls, float beginBias) {
    float m = 7.5f * PI;
    if (cls == 1) m *= 1.2f;
    else if (cls == 2) m *= 1.6f;
    return (0.3f + 0.7f * (1.0f - beginBias)) * m;
}
HD float JointSpeed(float dot, int dtMs) {
    return 2.0f * libm::acosf(Clamp(dot, -1.0f, 1.0f)) / ((float)dtMs * 0.001f);
}

// Each node takes the last history entry of its body part or appends one, in node order. Only
// with `append` are the new entries written; without it the plan is the same, for lanes that share
// the humanoid with one that appends.
HD void ApplyPrepare(const Ctx &c, const Anim &a, Humanoid &h, bool smooth, int frame, ApplyPlan &plan,
                     bool append = true) {
    plan.beginBias = smooth ? SmoothBeginBias(frame) : 0.0f;
    if (a.nodeCount > kBodyParts) Fatal("an animation moves more body parts than a humanoid has");
    if (!smooth) return;
    auto &hist = h.movementHistory;
    int16_t last[kBodyParts];
    for (int b = 0; b < kBodyParts; b++) last[b] = -1;
    const int entries = hist.count;
    for (int i = 0; i < entries; i++) {
        int32_t b = hist[i].nodeName;
        if (b >= 0 && b < kBodyParts) last[b] = (int16_t)i;
    }
    int count = entries;
    for (int n = 0; n < a.nodeCount; n++) {
        int bp = c.T().nodes[a.nodeFirst + n].bodyPart;
        int found = last[bp];
        plan.isNew[n] = found < 0;
        if (found < 0) {
            if (append) {
                MovementHistoryEntry e;
                memset(&e, 0, sizeof(e));
                e.nodeName = bp;
                e.timeDifferenceMs = 10;
                hist.push_back(e);
            }
            // A full history keeps its count (the append fails), and the node takes its last entry.
            found = count < hist.kCapacity ? count++ : count - 1;
        }
        plan.entry[n] = (int16_t)found;
    }
}

// A node's pose for the frame before smoothing: halfway between `frame` and the next (from the
// pose table while it lasts), the root's position turned by the humanoid's angle (only its height
// kept for a plan that carries the position), the body turned by that angle, and the node's pose
// offset blended in (the offset's stored orientation is first moved into the pose's neighbourhood,
// as GRF does in place). Returns the table entry while the orientation is still its halfway pose.
HD const MiddleEntry *NodeFramePose(const Ctx &c, const Anim &a, const NodeAnim &na, int frame, float baseRot, bool noPos,
                                    BiasedOffset &offset, Quat &ori, Vec3 &pos) {
    const int bp = na.bodyPart;
    const MiddleEntry *middle = nullptr;
    if (frame >= 0 && frame + 1 < na.interpFrames) {
        middle = &c.T().middle[na.interpFirst + frame * na.interpStride];
        ori = middle->orientation;
        pos = middle->position;
    } else {
        Quat oa, ob;
        Vec3 pa, pb;
        Interpolated(c, a, na, frame, oa, pa);
        Interpolated(c, a, na, frame + 1, ob, pb);
        BlendFrames(oa, pa, ob, pb, 0.5f, ori, pos);
    }
    if (bp == kBpPlayer) {
        if (noPos) {
            pos.v[0] = 0;
            pos.v[1] = 0;
        } else {
            pos.Rotate2D(baseRot);
        }
    }
    if (bp == kBpBody) {
        Quat rz;
        rz.SetAngleAxis(baseRot, Vec3(0, 0, 1));
        ori = rz * ori;
        ori.Normalize();
        middle = nullptr;
    }
    if (offset.bias != 0.0) {
        offset.orientation.MakeSameNeighborhood(ori);
        ori = ori.Lerp(offset.bias, offset.orientation).Normalized();
        middle = nullptr;
    }
    return middle;
}
// The slerp by `bias` from the table's normalized halfway pose toward `current` when the bias is
// zero and the table marks the pose as one whose zeros normalizing keeps: each nonzero element is
// kept and each zero takes the sign of a sum of two zeros. False when the shortcut does not apply.
HD bool SteadySlerp(const MiddleEntry *middle, const Quat &current, float bias, Quat &ori) {
    if (!(middle && middle->normalizedKeepsZeros && bias == 0.0f)) return false;
    const Quat &from = middle->orientation;
    Quat target = current;
    float cosHalf = from.q[3] * target.q[3] + from.q[0] * target.q[0] + from.q[1] * target.q[1] + from.q[2] * target.q[2];
    if (cosHalf < 0) {
        target = -target;
        cosHalf = -cosHalf;
    }
    if (fabsf(cosHalf) >= 1.0f) {
        ori = middle->normalized;
        return true;
    }
    if (!(fabsf(cosHalf) < 1.0f)) return false;
    for (int k = 0; k < 4; k++) {
        const float own = middle->normalized.q[k];
        ori.q[k] = own != 0.0f ? own : (SignBit(own) && SignBit(target.q[k]) != SignBit(bias)) ? -0.0f : 0.0f;
    }
    return true;
}
// A joint eases from its current rotation toward the frame's by the smoothing bias, and turns at
// most its joint class's speed (7.5 pi rad/s; elbows and knees 1.2 times, ankles 1.6 times; 30% of
// it at the start of an animation).
HD void SmoothJoint(Quat &ori, const Quat &current, const MiddleEntry *middle, int bp, float beginBias, float bias, int dtMs) {
    if (!SteadySlerp(middle, current, bias, ori)) ori = ori.Slerp(bias, current).Normalized();
    const float dot = ori.MakeSameNeighborhood(current);
    const float most = JointSpeedLimit(JointSpeedClass(bp), beginBias);
    const float speed = JointSpeed(dot, dtMs);
    if (speed > most) {
        const Quat wanted = current.RotationTo(ori).Normalized();
        ori = (wanted.RotationMultipliedBy(most / speed) * current).Normalized();
    }
}
// At the start of an animation the root's height eases toward its current height and rises or
// falls at most 2.8 m/s (6 m/s into a special state).
HD void SmoothRootHeight(Vec3 &pos, const Vec3 &current, const Vec3 &basePos, float beginBias, float bias, bool special, int dtMs) {
    pos.v[2] = pos.v[2] * (1.0f - bias) + current.v[2] * bias;
    const float allowed = (special ? 6.0f : 2.8f) * ((float)dtMs * 0.001f);
    float height = pos.v[2] + basePos.v[2];
    const float wanted = fabsf(height - current.v[2]);
    float share = 1.0f;
    if (wanted > allowed) share = allowed / wanted;
    height = (height * share + current.v[2] * (1.0f - share)) * beginBias + height * (1.0f - beginBias);
    pos = pos.Get2D() + Vec3(0, 0, height);
}
// One node of a humanoid's frame: its pose, smoothed against the movement history (a node new to
// the history starts it at this pose), then written to the node.
HDN void ApplyNode(LocalRef<const Ctx> context, GlobalRef<const Anim> animation, GlobalRef<const Skeleton> skeleton, GlobalRef<Humanoid> humanoid, int ni, int frame, bool smooth,
                   float smoothFactor, Vec3 basePos, float baseRot, GlobalPointer<BiasedOffset> offsets, int dtMs, bool noPos,
                   GlobalRef<const ApplyPlan> applyPlan) {
    const Ctx &c = context;
    const ApplyPlan &plan = applyPlan;
    const Anim &a = animation;
    const Skeleton &sk = skeleton;
    Humanoid &h = humanoid;
    const NodeAnim &na = c.T().nodes[a.nodeFirst + ni];
    const int bp = na.bodyPart;
    NodeState &node = h.nodes[sk.nodeMap[bp]];
    Quat ori;
    Vec3 pos;
    const MiddleEntry *middle = NodeFramePose(c, a, na, frame, baseRot, noPos, offsets[bp], ori, pos);
    if (smooth) {
        MovementHistoryEntry &e = h.movementHistory[plan.entry[ni]];
        if (plan.isNew[ni]) {
            e.position = pos;
            e.orientation = ori;
        }
        const float beginBias = plan.beginBias;
        const float bias = 0.0f + beginBias * smoothFactor * 0.5f;
        if (bp != kBpPlayer) {
            Quat current = node.rotation;
            current.MakeSameNeighborhood(e.orientation);
            if (dtMs > 0) SmoothJoint(ori, current, middle, bp, beginBias, bias, dtMs);
            e.orientation = current;
        } else {
            const Vec3 current = node.position;
            if (dtMs > 0 && beginBias > 0.01f) SmoothRootHeight(pos, current, basePos, beginBias, bias, a.outgoingSpecialState != kStrEmpty, dtMs);
            e.position = current;
        }
        e.timeDifferenceMs = dtMs;
    }
    if (bp != kBpPlayer) {
        ori.MakeSameNeighborhood(node.rotation);
        node.rotation = ori;
    } else {
        node.position = pos + basePos;
    }
}

// Applies the buffered frame of the active players and the officials; humanoids are independent.
HDN void FetchPutBuffers(GlobalRef<World> world, LocalRef<const Ctx> context, uint32_t active) {
    World &w = world;
    const Ctx &c = context;
    const PlayerSet players{active};
    const int playing = players.size(), count = playing + 3;
    // Humanoid k's place in the state: the players', then the officials'.
    auto place = [&](int k) { return k < playing ? players[k] : w.match.playerCount + k - playing; };
    auto humanoid = [&](int k) -> Humanoid & {
        return k < playing ? w.match.players[players[k]].base.humanoid : w.match.officials[k - playing].humanoid;
    };
    // A humanoid's pose reads and writes only its own state, and a node only its own body part's
    // node, offset and history entry.
    ApplyPlan *const plans = c.ws->applyPlans;
    auto applyNode = [&](int k, int n) {
        Humanoid &h = humanoid(k);
        AnimApplyBuffer &buf = h.applyBuf;
        const Anim &a = c.A(buf.anim);
        if (n < a.nodeCount)
            ApplyNode(c, a, c.skeletons[place(k)], h, n, buf.frameNum, buf.smooth, buf.smoothFactor, buf.position, buf.orientation.value(),
                      buf.offsets, 10, buf.noPos, plans[k]);
    };
    auto prepare = [&](int k, bool append) {
        Humanoid &h = humanoid(k);
        ApplyPrepare(c, c.A(h.applyBuf.anim), h, h.applyBuf.smooth, h.applyBuf.frameNum, plans[k], append);
    };
    if constexpr (kGroupLanes >= 16) {
        // A group of 16 lanes or more leaves most lanes idle when each takes a humanoid (25 of 64
        // lanes for 14 rounds, 13 in 5-a-side), so the lanes prepare a humanoid each and then take
        // the nodes of all of them in turn: 6 rounds on 64 lanes, 11 on 32 and 22 on 16 (28 before).
        // Measured, ms per step: one match of 64 lanes 13.8 -> 13.3, 1,024 of 5-a-side (64) 27.6 -> 26.3,
        // 4,096 (32) 47.2 -> 45.7, 8,192 (16) 82.3 -> 79.6.
        for (int k = GroupRank(); k < count; k += kGroupLanes) prepare(k, true);
        GroupSync();
        for (int u = GroupRank(); u < count * kBodyParts; u += kGroupLanes) applyNode(u / kBodyParts, u % kBodyParts);
    } else {
        // The lanes take the humanoids in turn; the humanoids left over after the whole rounds have
        // their nodes split over the lanes instead, when that at least halves the rounds those
        // humanoids take.
        constexpr int kNodeRounds = (kBodyParts + kGroupLanes - 1) / kGroupLanes;
        int whole = count;
        if (2 * (count % kGroupLanes) * kNodeRounds <= kBodyParts) whole = count - count % kGroupLanes;
        for (int k = GroupRank(); k < whole; k += kGroupLanes) {
            prepare(k, true);
            for (int n = 0; n < kBodyParts; n++) applyNode(k, n);
        }
        for (int k = whole; k < count; k++) {
            prepare(k, GroupRank() == 0);
            GroupSync();
            for (int n = GroupRank(); n < kBodyParts; n += kGroupLanes) applyNode(k, n);
        }
    }
    GroupSync();
}

// ---- spatial state --------------------------------------------------------------------------------
// The body directions allowed relative to movement, and the zero vector last.
HD Vec3 AllowedBodyDir(int i) {
    const float s = 0x1.6a09e6p-1f;
    switch (i) {
        case 0:
            return Vec3(0, -1, 0);
        case 1:
            return Vec3(-s, -s, 0);
        case 2:
            return Vec3(s, -s, 0);
        case 3:
            return Vec3(-s, s, 0);
        case 4:
            return Vec3(s, s, 0);
    }
    return Vec3(0, 0, 0);
}
// Angle2D(Vec3(0,-1,0)) of each allowed direction: the first is -0, the last +0.
HD float AllowedBodyDirAngle(int i) {
    switch (i) {
        case 0:
            return -0.0f;
        case 1:
            return -0x1.921fb6p-1f;
        case 2:
            return 0x1.921fb6p-1f;
        case 3:
            return -0x1.2d97c8p+1f;
        case 4:
            return 0x1.2d97c8p+1f;
    }
    return 0.0f;
}
constexpr int kNoAllowedBodyDirection = 5;
HDN int BodyDirectionIndex(Vec3 src) {
    float best = -1.0f;
    int bi = kNoAllowedBodyDirection;
    for (int i = 0; i < 5; i++) {
        float d = AllowedBodyDir(i).Dot(src);
        if (d > best) {
            best = d;
            bi = i;
        }
    }
    return bi;
}

// Ground-plane movement in m/s at `frame` of a position list of two frames or more.
HDN Vec3 MovementAtFrame(GlobalPointer<const Vec3> pos, int count, uint32_t frame, uint32_t smooth) {
    if (frame == (uint32_t)(count - 1)) return (pos[count - 1] - pos[count - 2]).Get2D() * 100.0f;
    if (frame == 0) return (pos[1] - pos[0]).Get2D() * 100.0f;
    Vec3 total;
    uint32_t n = 0;
    for (int f = (int)(frame - smooth); f <= (int)(frame + smooth); f++) {
        if (f > 0 && f < count) {
            total += (pos[f] - pos[f - 1]).Get2D() * 100.0f;
            n++;
        }
    }
    if (n > 0) total /= Vec3((float)n);
    return total;
}

// Where the humanoid stands at its animation's current frame: the planned position while the
// plan lasts, else the animation's root (on the ground) turned by the start angle; plus the
// smuggle offsets.
HD Vec3 FramePosition(const Ctx &c, const Humanoid &h, const Anim &a) {
    const AnimationState &cur = h.anim;
    if ((uint32_t)cur.positions.count > (uint32_t)cur.frameNum)
        return h.startPos + cur.positions[cur.frameNum] + cur.actionSmuggleOffset + cur.actionSmuggleSustainOffset +
               cur.movementSmuggleOffset;
    Quat o;
    Vec3 root;
    GetKeyFrame(c, a, kBpPlayer, cur.frameNum, o, root);
    root.v[2] = 0.0f;
    return h.startPos + root.Rotated2D(h.startAngle.value()) + cur.actionSmuggleOffset + cur.actionSmuggleSustainOffset +
           cur.movementSmuggleOffset;
}
// The body direction relative to the movement, for a moving humanoid: the body's angle off the
// movement, held within 0.12 pi at a sprint (from 0.125 pi) and 0.495 pi walking (from half a
// turn); `unsnapped` is that angle before it snaps to the allowed directions.
HD Vec3 RelativeBody(const Vec3 &body, float angle, int velocityCat, float &unsnapped) {
    Vec3 rel = body.Rotated2D(-angle);
    const float off = rel.Angle2D(Vec3(0, -1, 0));
    unsnapped = off;
    if (velocityCat == kVelSprint && fabsf(off) >= 0.125f * PI) {
        rel = Vec3(0, -1, 0).Rotated2D(0.12f * PI * SignSide(off));
        unsnapped = rel.Angle2D(Vec3(0, -1, 0));
    } else if (velocityCat == kVelWalk && fabsf(off) >= 0.5f * PI) {
        rel = Vec3(0, -1, 0).Rotated2D(0.495f * PI * SignSide(off));
        unsnapped = rel.Angle2D(Vec3(0, -1, 0));
    }
    return rel;
}
// A humanoid's spatial state for the tick (GRF's humanoid spatial state), from its own animation
// and last position only: position; the actual
// movement since the last tick, less the smuggles' and half the offset's movement (the physics
// movement, which is the movement); the animation's own movement; velocity and its category;
// the direction (the movement's, or the body's when idle) and angle; the body direction relative
// to it, snapped to the allowed directions, and in the world.
HDN SpatialState NextSpatialState(LocalRef<const Ctx> context, GlobalRef<const Humanoid> humanoid) {
    const Ctx &c = context;
    const Humanoid &h = humanoid;
    ENG_SCOPE(29);
    const AnimationState &cur = h.anim;
    const Anim &a = c.A(cur.anim);
    SpatialState s = h.spatial;
    const Vec3 position = FramePosition(c, h, a);
    if (cur.frameNum > 12) s.foot = a.outgoingFoot;
    s.actualMovement = (position - h.prevPosition2D) * 100.0f;
    s.physicsMovement = s.actualMovement - (s.actionSmuggleMovement) - (s.movementSmuggleMovement) - (s.positionOffsetMovement * 0.5f);
    s.animationMovement = s.physicsMovement;
    if (cur.positions.count > 0)
        s.animationMovement = MovementAtFrame(c.T().positions + a.posFirst, a.posCount, cur.frameNum, 1).Rotated2D(h.startAngle.value());
    s.movement = s.physicsMovement;
    Vec3 bodyPos;
    Quat bodyOri;
    float bodyTurn;
    GetKeyFrameZ(c, a, kBpBody, cur.frameNum, bodyOri, bodyPos, bodyTurn);
    const Vec3 body = Vec3(0, -1, 0).Rotated2D(bodyTurn + h.startAngle.value() + cur.rotationSmuggleOffset.value());
    s.floatVelocity = s.movement.Length();
    s.velocityCat = VelocityCat(s.floatVelocity);
    s.directionVec = s.velocityCat != kVelIdle ? s.movement.Normalized() : body;
    s.position = position;
    s.angle.set(ModulateIntoRange(-PI, PI, FixAngle(s.directionVec.Angle2D())));
    int snapped = 0;
    float unsnapped = AllowedBodyDirAngle(0);
    if (s.velocityCat != kVelIdle) {
        s.relBodyDirectionVecNonQuantized = RelativeBody(body, s.angle.value(), s.velocityCat, unsnapped);
        snapped = BodyDirectionIndex(s.relBodyDirectionVecNonQuantized);
    } else {
        s.relBodyDirectionVecNonQuantized = Vec3(0, -1, 0);
    }
    s.relBodyDirectionVec = AllowedBodyDir(snapped);
    s.relBodyAngle.set(AllowedBodyDirAngle(snapped));
    s.relBodyAngleNonQuantized.set(unsnapped);
    s.bodyDirectionVec = s.relBodyDirectionVec.Rotated2D(s.angle.value());
    s.bodyAngle.set(s.bodyDirectionVec.Angle2D(Vec3(0, -1, 0)));
    return s;
}

}  // namespace eng
