// The table as the collection rewrites it: pages of the virtual space are mapped as they are first
// written (HashTable::add_leaf_node / add_interior_node, hash_table.h:359-468). Whoever starts a page
// numbers it from poolTop (page 0 of the physical pool is never used, hash_table.h:821) unless the
// page is already mapped.
#pragma once

#include <hip/hip_runtime.h>

#include "hd_internal.h"

namespace hd {

struct TableRef {
    Geom g;
    uint32_t* vpool;
    uint32_t* page_table;
    uint32_t* bucket_sizes;
    uint32_t* pool_top;
    uint32_t pool_pages;
};

__device__ inline bool table_map_page(const TableRef& T, uint32_t page) {
    if (atomicCAS(&T.page_table[page], 0u, 0xFFFFFFFFu) != 0u) return true;  // mapped already
    const uint32_t phys = atomicAdd(T.pool_top, 1u);
    if (phys >= T.pool_pages) {
        atomicExch(&T.page_table[page], 0u);
        return false;
    }
    atomicExch(&T.page_table[page], phys);
    return true;
}

}  // namespace hd
