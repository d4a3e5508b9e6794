// HostStage under NoAlloc: growing it throws before any runtime call; memory
// that it holds stays usable.  Runs without a device.
#include <cstdio>

#include "dtb_engine.hpp"

int main()
{
    dtb::HostStage s;
    int code = -1;
    {
        dtb::devmem::NoAlloc no_alloc;
        try {
            s.reserve(64);
        } catch (const dtb::Error &e) {
            code = e.code;
        }
        if (s.reserve(0) != nullptr)
            return 1;
    }
    if (code != dtb::kInvalidParameter) {
        std::printf("reserve under NoAlloc: code %d\n", code);
        return 1;
    }
    std::puts("ok");
    return 0;
}
