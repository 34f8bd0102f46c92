// The shape that a chain to one destination takes (hcclx_internal.h, wide_shape_for), asked of the library on the CPU
// (tests/test_host_wide_shapes.py).  argv: compute units, 1 or 0 (whether LDS may hold workgroups off a CU), bytes of an element,
// sources, bytes by which every other source is off the destination's alignment, then the segments' elements.  Prints the shape and
// how many workgroups LDS leaves to a CU (0: it holds none off).
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "hcclx_internal.h"
#include "kernels/segtab.h"

int main(int argc, char **argv)
{
    const char *const names[] = {"many", "small", "three", "four", "large"};
    hcclx::DeviceCtx ctx;
    ctx.num_cus = std::atoi(argv[1]);
    ctx.wide_min_tiles = 2u * static_cast<uint32_t>(ctx.num_cus);
    ctx.fold_lds_hold = std::atoi(argv[2]) != 0;
    const int esz = std::atoi(argv[3]);
    std::vector<hcclx_wide_seg_t> segs;
    for (int k = 6; k < argc; ++k) {
        hcclx_wide_seg_t s = {};
        s.count = std::strtoull(argv[k], nullptr, 10);
        s.nsrc = static_cast<uint32_t>(std::atoi(argv[4]));
        s.ndst = 1;
        for (uint32_t q = 0; q < s.nsrc; ++q) s.src[q] = reinterpret_cast<const void *>((1ull << 40) * (q + 2) + (q & 1u) * std::atoi(argv[5]));
        s.dst[0] = reinterpret_cast<void *>(1ull << 40);
        segs.push_back(s);
    }
    uint32_t per_cu = 99;
    const hcclx::WideShape shape = hcclx::wide_shape_for(&ctx, segs.data(), static_cast<uint32_t>(segs.size()), esz, &per_cu);
    std::printf("%s %u\n", names[shape], per_cu);
    return 0;
}
