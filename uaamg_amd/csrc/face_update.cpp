// Host side of the device pressure-gradient update (face_update.h).
#include "face_update.h"

#include <algorithm>
#include <vector>

#include "leaf_match.h"
#include "leaf_topology.h"
#include "poisson_solver.h"

namespace uaamg {

namespace {

struct DevBuf {
    void* p = nullptr;
    void release() {
        if (p) (void)hipFree(p);
        p = nullptr;
    }
    ~DevBuf() { release(); }
};

}  // namespace

int apply_pressure_gradient_device(PoissonDevice& d, const float* pressure_dev, const FaceGridRef* grids,
                                   FaceChannelRef* channels, float dt, float friction, bool values_on_device,
                                   std::string& err) {
    if (!d.on_device()) {
        err = "handle was created without a device (device < 0)";
        return -4;
    }
    hipStream_t s = d.stream();
    if (hipSetDevice(d.device()) != hipSuccess) {
        err = "hipSetDevice failed";
        return -3;
    }
    if (d.follow_caller()) {
        err = d.error();
        return -3;
    }
    auto hip_fail = [&](hipError_t e, const char* what) {
        err = std::string(what) + ": " + hipGetErrorString(e);
        (void)hipStreamSynchronize(s);
        return -3;
    };
    const PoissonLevelHost& l0 = d.host().levels[0];
    // inputs: liquid phi, face weights, solid velocity
    const char* names[3] = {"liquid_phi", "face_weights", "solid_velocity"};
    LeafMatch match;
    int in_set[3], ch_set[3];
    DevBuf in_buf[3];
    const float* in_dev[3] = {nullptr, nullptr, nullptr};
    for (int g = 0; g < 3; ++g) {
        const FaceGridRef& r = grids[g];
        in_set[g] = match.add(r.nleaf, r.origins);
        if (r.nleaf == 0) continue;
        if (values_on_device) {
            in_dev[g] = r.values;
            continue;
        }
        const size_t bytes = size_t(r.nleaf) * kLeafSize * size_t(r.ncomp) * sizeof(float);
        if (hipError_t e = hipMalloc(&in_buf[g].p, bytes)) return hip_fail(e, "hipMalloc");
        if (hipError_t e = hipMemcpyAsync(in_buf[g].p, r.values, bytes, hipMemcpyHostToDevice, s))
            return hip_fail(e, "upload grid values");
        in_dev[g] = static_cast<const float*>(in_buf[g].p);
    }
    const LevelView& v0 = d.level_view(0);
    int64_t most = 0;
    for (int c = 0; c < 3; ++c) {
        ch_set[c] = match.add(channels[c].nleaf, channels[c].origins);
        most = std::max(most, channels[c].nleaf);
    }
    static_assert(sizeof(Coord) == 12, "origins are matched as triples of int32");
    const int dof = match.add(int64_t(l0.nleaf()), l0.nleaf() ? &l0.origin[0].x : nullptr);
    // the channels' leaf tables and masks in the handle's grow-only buffer (a repeated call allocates nothing)
    const size_t tab_bytes = (size_t(most) * kGradTab * sizeof(int32_t) + 255) & ~size_t(255);
    const size_t act_bytes = size_t(most) * 8 * sizeof(uint64_t);
    char* aux = static_cast<char*>(d.aux(match.bytes() + 3 * (tab_bytes + act_bytes)));
    if (!aux) return hip_fail(hipErrorOutOfMemory, "device scratch");
    auto tab_at = [&](int c) { return reinterpret_cast<int32_t*>(aux + match.bytes() + size_t(c) * tab_bytes); };
    auto act_at = [&](int c) {
        return reinterpret_cast<uint64_t*>(aux + match.bytes() + 3 * tab_bytes + size_t(c) * act_bytes);
    };
    if (hipError_t e = match.build(aux, s)) return hip_fail(e, "leaf match");
    // refused origins are found before any channel is touched
    int32_t bad = -1;
    if (hipError_t e = hipMemcpyAsync(&bad, match.bad(), sizeof(bad), hipMemcpyDeviceToHost, s))
        return hip_fail(e, "leaf match");
    if (hipError_t e = hipStreamSynchronize(s)) return hip_fail(e, "leaf match sync");
    if (bad >= 0) {
        const char* what = names[0];
        bool misaligned = false;
        for (int g = 0; g < 6; ++g) {
            const int64_t n = g < 3 ? grids[g].nleaf : channels[g - 3].nleaf;
            what = g < 3 ? names[g] : "velocity channel";
            if (bad_origins(n, g < 3 ? grids[g].origins : channels[g - 3].origins, &misaligned)) break;
        }
        err = std::string(what) + (misaligned ? ": leaf origin not a multiple of 8" : ": duplicate leaf origins");
        return -1;
    }
    DevBuf vel_b, upd_b, refl_b;   // values held on the host: one channel's at a time
    auto download = [&](int c) -> int {
        FaceChannelRef& ch = channels[c];
        const size_t n = size_t(ch.nleaf), vbytes = n * kLeafSize * sizeof(float);
        if (n == 0) return 0;
        if (hipError_t e = hipMemcpyAsync(ch.active, act_at(c), n * 8 * sizeof(uint64_t), hipMemcpyDeviceToHost, s))
            return hip_fail(e, "download active masks");
        if (values_on_device) return 0;
        if (hipError_t e = hipMemcpyAsync(ch.values, vel_b.p, vbytes, hipMemcpyDeviceToHost, s))
            return hip_fail(e, "download velocity");
        if (ch.update)
            if (hipError_t e = hipMemcpyAsync(ch.update, upd_b.p, vbytes, hipMemcpyDeviceToHost, s))
                return hip_fail(e, "download update");
        if (ch.reflected)
            if (hipError_t e = hipMemcpyAsync(ch.reflected, refl_b.p, vbytes, hipMemcpyDeviceToHost, s))
                return hip_fail(e, "download reflected");
        if (hipError_t e = hipStreamSynchronize(s)) return hip_fail(e, "pressure gradient sync");
        for (DevBuf* b : {&vel_b, &upd_b, &refl_b}) b->release();
        return 0;
    };
    // A channel's masks are read after those of the channels before it are written, where the arrays overlap.
    int pending = 0;   // first channel whose masks are still to be downloaded
    auto shares_masks = [&](int c) {
        auto first = [&](int k) { return reinterpret_cast<uintptr_t>(channels[k].active); };
        auto end = [&](int k) { return first(k) + size_t(channels[k].nleaf) * 8 * sizeof(uint64_t); };
        for (int k = pending; k < c; ++k)
            if (first(k) < end(c) && first(c) < end(k)) return true;
        return false;
    };
    for (int c = 0; c < 3; ++c) {
        FaceChannelRef& ch = channels[c];
        if (ch.nleaf == 0) continue;
        if (values_on_device && shares_masks(c)) {
            for (; pending < c; ++pending)
                if (int rc = download(pending)) return rc;
            if (hipError_t e = hipStreamSynchronize(s)) return hip_fail(e, "pressure gradient sync");
        }
        int32_t* const tab_d = tab_at(c);
        uint64_t* const act_d = act_at(c);
        const size_t n = size_t(ch.nleaf);
        const size_t vbytes = n * kLeafSize * sizeof(float);
        const int here[3] = {0, 0, 0}, low[3] = {c == 0 ? -8 : 0, c == 1 ? -8 : 0, c == 2 ? -8 : 0};
        std::vector<MatchColumn> cols(kGradTab);
        auto column = [&](int at, int set, const int* o) { cols[size_t(at)] = {set, {o[0], o[1], o[2]}}; };
        column(kGradPhi, in_set[0], here);
        column(kGradPhiLow, in_set[0], low);
        column(kGradDof, dof, here);
        column(kGradDofLow, dof, low);
        column(kGradW, in_set[1], here);
        column(kGradSolid, in_set[2], here);
        if (hipError_t e = match.query(ch_set[c], cols, tab_d, s)) return hip_fail(e, "leaf match");
        if (hipError_t e = hipMemcpyAsync(act_d, ch.active, n * 8 * sizeof(uint64_t), hipMemcpyHostToDevice, s))
            return hip_fail(e, "upload active masks");
        float* vel = ch.values;
        float* upd = ch.update;
        float* refl = ch.reflected;
        if (!values_on_device) {
            if (hipError_t e = hipMalloc(&vel_b.p, vbytes)) return hip_fail(e, "hipMalloc");
            if (hipError_t e = hipMemcpyAsync(vel_b.p, ch.values, vbytes, hipMemcpyHostToDevice, s))
                return hip_fail(e, "upload velocity");
            vel = static_cast<float*>(vel_b.p);
            if (ch.update) {
                if (hipError_t e = hipMalloc(&upd_b.p, vbytes)) return hip_fail(e, "hipMalloc");
                upd = static_cast<float*>(upd_b.p);
            }
            if (ch.reflected) {
                if (hipError_t e = hipMalloc(&refl_b.p, vbytes)) return hip_fail(e, "hipMalloc");
                refl = static_cast<float*>(refl_b.p);
            }
        }
        GradArgs a{};
        a.tab = tab_d;
        a.phi = in_dev[0];
        a.w = in_dev[1];
        a.sv = in_dev[2];
        a.pressure = pressure_dev;
        a.dmask = v0.mask;
        a.dofbase = v0.dofbase;
        a.phi_bg = grids[0].bg[0];
        for (int k = 0; k < 3; ++k) {
            a.w_bg[k] = grids[1].bg[k];
            a.sv_bg[k] = grids[2].bg[k];
        }
        a.channel = c;
        a.dt = dt;
        a.dx = l0.dx;
        a.friction = friction;
        if (hipError_t e = launch_pressure_gradient(ch.nleaf, a, act_d, vel, upd, refl, s))
            return hip_fail(e, "pressure gradient kernel");
        if (!values_on_device)
            if (int rc = download(c)) return rc;
    }
    // values on the device: a channel's masks are uploaded beside the kernel of the one before
    if (values_on_device)
        for (; pending < 3; ++pending)
            if (int rc = download(pending)) return rc;
    if (hipError_t e = hipStreamSynchronize(s)) return hip_fail(e, "pressure gradient sync");
    return 0;
}

}  // namespace uaamg
