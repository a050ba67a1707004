// The key of a batch's captured frame: settings that launch different grids give
// different keys, and the same settings the same key.
#include <cstdio>

#include "oibvh_batch.cpp"

static bool same(const oibvh_batch& b, uint32_t blocks0, uint32_t blocks1)
{
    uint64_t k0[8], k1[8];
    b.ctx->trav_blocks = blocks0;
    detect_key(&b, 0, k0);
    b.ctx->trav_blocks = blocks1;
    detect_key(&b, 0, k1);
    return std::memcmp(k0, k1, sizeof k0) == 0;
}

int main()
{
    static oibvh_ctx c;
    c.cus = 256;
    static oibvh_batch b;
    b.ctx = &c;
    b.desc_gen = 3;
    const uint32_t per_cu4 = 4u * 256u;
    int bad = 0;
    auto expect = [&](bool ok, const char* what) {
        if (!ok) std::printf("wrong: %s\n", what), bad = 1;
    };
    // 0 launches six workgroups per CU for some steps, 1024 four for all
    expect(!same(b, 0, per_cu4), "0 and four workgroups per CU share a key");
    expect(!same(b, 0, 1), "0 and 1");
    expect(!same(b, 2048, 4096), "2048 and 4096");
    for (uint32_t v : {0u, 1u, per_cu4, 8192u}) expect(same(b, v, v), "one setting has two keys");
    return bad;
}
