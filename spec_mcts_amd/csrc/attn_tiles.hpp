// What smh_shared_prefix_attn_qkv_tiles asks of its tensors: the entry point refuses others, a decode layer has other launches for them.
#pragma once

#include <initializer_list>

#include "smh_common.hpp"

namespace smh {

struct TileTensors {
    const void *slabs, *out, *cos_tab, *sin_tab, *prompt_k, *prompt_v, *cache_k, *cache_ks, *cache_v, *cache_vs;
    long B, H, Hkv, P;
    long cache_rows;         // of the pool that a page table points to, else of all branches
};

// Queries of a workgroup: eight while those fill one round of compute units, else 16 (us, 16 and 8: 32 heads, 64 branches after 512 rows 24.4 and
// 19.4, 17 20.5 and 14.2, 100, two rounds of eight, 24.1 and 30.6; 64 heads over 8, 30 branches after 2047 rows 26.3 and 23.7, 100 48.8 and 76.3)
inline int attn_tile_queries(long Bq, long Hkv) { return Hkv * ((Bq + 7) / 8) <= 256 ? 8 : 16; }

// Why it does not take them; nullptr: it does
inline const char *attn_tiles_refuse(const TileTensors &t) {
    auto aligned = [](std::initializer_list<const void *> list, uintptr_t to) {
        for (const void *x : list)
            if ((uintptr_t)x % to != 0) return false;
        return true;
    };
    if (!aligned({t.slabs, t.prompt_k, t.prompt_v}, 16)) return "the slabs and the prefix must be 16-byte aligned";
    if (!aligned({t.out, t.cos_tab, t.sin_tab, t.cache_k, t.cache_v}, 8)) return "out, the rotation tables and the cache codes must be 8-byte aligned";
    if (!aligned({t.cache_ks, t.cache_vs}, 4)) return "the cache scales must be 4-byte aligned";
    if (t.P * t.Hkv * 256 >= 1L << 32) return "the prefix exceeds 32-bit offsets";
    if (t.cache_rows < 0 || t.cache_rows >= 1L << 31 || t.cache_rows * t.Hkv * 64 >= 1L << 32) return "the cache exceeds 32-bit offsets";
    const long Bq = t.B * (t.H / t.Hkv), qt = attn_tile_queries(Bq, t.Hkv);
    if ((Bq + qt - 1) / qt > 65535 || t.Hkv > 8 * 65535) return "more tiles of queries or heads than a grid has";
    return nullptr;
}

}  // namespace smh
