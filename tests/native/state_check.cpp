// State of an instance read and written where no device memory may be taken
// (NoAlloc) against the same through device memory: 70,003 neurons, three
// pieces of the pinned memory.
#include <cstdio>
#include <cstring>
#include <memory>

#include "dtb_engine.hpp"

namespace {
constexpr uint32_t kN = 70003;

struct State {
    std::vector<float> V = std::vector<float>(kN), iou = V, J = std::vector<float>(4 * (size_t)kN), isyn = V;
    std::vector<int32_t> t = std::vector<int32_t>(kN);
    std::vector<uint8_t> f = std::vector<uint8_t>(kN), emitted = f;

    void read(dtb::Engine &e, int id)
    {
        e.settle();
        e.get(id)->read_state(e.call_stage(), V.data(), t.data(), f.data(), emitted.data(), iou.data(), J.data(),
                              isyn.data(), e.stream());
    }
    void write(dtb::Engine &e, int id) const
    {
        e.get(id)->write_state(e.call_stage(), V.data(), t.data(), f.data(), iou.data(), J.data(), e.stream());
    }
    bool same(const State &o) const
    {
        auto eq = [](const auto &a, const auto &b) { return std::memcmp(a.data(), b.data(), a.size() * sizeof(a[0])) == 0; };
        return eq(V, o.V) && eq(t, o.t) && eq(f, o.f) && eq(emitted, o.emitted) && eq(iou, o.iou) && eq(J, o.J) &&
               eq(isyn, o.isyn);
    }
};
}  // namespace

int main()
{
    try {
        dtb::Engine e(0);
        dtb::FanoutSpec spec;
        spec.n = kN;
        spec.K = 60;
        spec.net_seed = 7;
        const float g[4] = {0.01f, 0.0005f, 0.1f, 0.005f};
        std::memcpy(spec.g_ui, g, sizeof(g));
        const int id = e.add(std::make_unique<dtb::Instance>(spec, 0.1f, 5, e.admit_stream()));
        const uint32_t pops[2] = {0, 1};
        const float mean[2] = {3.0f, 3.0f}, sd[2] = {0.1f, 0.1f}, tau[2] = {4.0f, 4.0f};
        e.get(id)->set_ou(pops, mean, sd, tau, 2, e.admit_stream());
        e.get(id)->configure_run(1, true, e.admit_stream());
        e.mark_dirty();
        (void)e.call_stage().reserve(dtb::kCallStageBytes);
        State first, a, b;
        first.read(e, id);
        e.run(200, 0);
        a.read(e, id);
        {
            dtb::devmem::NoAlloc no_alloc;
            b.read(e, id);
        }
        if (!a.same(b) || a.same(first)) {
            std::puts("read differs");
            return 1;
        }
        e.run(50, 0);
        e.settle();
        {
            dtb::devmem::NoAlloc no_alloc;
            a.write(e, id);
        }
        b.read(e, id);
        b.emitted = a.emitted;   // (not written)
        std::puts(a.same(b) ? "ok" : "write differs");
        return 0;
    } catch (const std::exception &x) {
        std::printf("error: %s\n", x.what());
        return 1;
    }
}
