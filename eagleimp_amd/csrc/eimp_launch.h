// eimp_launch.h -- kernel launchers, between the device code and the engine.
#pragma once

#include "eimp_internal.h"

namespace eimp {

// raises a kernel's dynamic-LDS limit (process-wide; never lowered)
hipError_t raise_lds_limit(const void *fn, size_t lds);

// pieces of device arrays for k_gather: piece i, bytes[i] (a multiple of 4) from
// src[i], goes to off[i] (a multiple of 16) of the destination
constexpr uint32_t kGatherPieces = 24;
struct GatherArgs {
    const void *src[kGatherPieces];
    uint32_t off[kGatherPieces], bytes[kGatherPieces];
    uint32_t n;
};
// dst: pinned host memory as the device sees it
hipError_t launch_gather(const GatherArgs &a, void *dst, hipStream_t s);

hipError_t launch_site_to_hap(const PanelDev &P, uint64_t *hap, hipStream_t s);
hipError_t launch_panel_mono(const PanelDev &P, uint64_t *pand, uint64_t *por, hipStream_t s);
hipError_t launch_distance(const PanelDev &P, const TgtDev *tg, const uint32_t *tlist,
                           uint32_t nsel, hipStream_t s);
hipError_t launch_select(const PanelDev &P, const TgtDev *tg, uint32_t n, hipStream_t s);
hipError_t launch_monos(const PanelDev &P, const TgtDev *tg, const uint32_t *tlist, uint32_t n,
                        uint32_t max_ww, uint32_t ncu, hipStream_t s);
hipError_t launch_splits(const PanelDev &P, const TgtDev *tg, uint32_t n, hipStream_t s);
hipError_t launch_bits_to_list(const TgtDev *tg, uint32_t n, uint32_t nbits_bh, int which,
                               hipStream_t s);
hipError_t launch_cref(const PanelDev &P, const TgtDev *tg, const CrefItem *items, uint32_t nitems,
                       uint32_t maxK, bool ident, hipStream_t s);
uint32_t cref_max_k();
hipError_t launch_digest_count0(const TgtDev *tg, uint32_t n, hipStream_t s);
hipError_t launch_cref_rows(const TgtDev *tg, uint32_t t, uint32_t Mp, uint64_t *rows, uint32_t rw,
                            hipStream_t s);
hipError_t launch_digest_rows(const TgtDev *tg, const uint32_t *d_n, uint32_t nmax, uint64_t *dig,
                              hipStream_t s);
size_t pbwt_big_lds_bytes(uint32_t K);
uint32_t pbwt_big_max_k();
hipError_t launch_pbwt_big(const BigItem *items, uint32_t nitems, uint32_t maxK, hipStream_t s);
int pbwt_variant_count();
int pbwt_variant_threads(int v);
int pbwt_variant_cpw(int v);
uint32_t pbwt_variant_maxk(int v);
size_t pbwt_lds_bytes(int v, uint32_t Kpad);
// occ (or null): resident workgroups per CU
hipError_t pbwt_prepare(int v, size_t lds, int *occ);
// chain items (CHAIN_ROWS ones, or the other kinds): grid workgroups, one item
// each, or with ctr taking items in turn up to *d_items; starts: for
// CHAIN_STARTS items
hipError_t launch_order(int v, const TgtDev *tg, const OrderItem *items, bool rows, uint32_t grid,
                        const uint32_t *d_items, uint32_t *ctr, uint16_t *starts, size_t lds,
                        hipStream_t s);
// the rows of one forward chain from the starts, and the order after each
hipError_t launch_dense(int v, const TgtDev *tg, uint32_t nblk, const uint16_t *starts, int32_t *absperm,
                        size_t lds, hipStream_t s);
// rows: pref = prefix sums of pbwt_blocks over the targets, n + 1 (n = *d_n if
// d_n is given); blocks = their sum or an upper bound; list: room for twice
// their sum, cnt: kRowsCounters words, zero
hipError_t launch_rows(const TgtDev *tg, const uint32_t *d_n, uint32_t n, const uint32_t *pref,
                       RowItem *list, uint32_t *cnt, uint32_t Kpad, uint64_t blocks, uint32_t ncu,
                       hipStream_t s);
hipError_t launch_prep_dev(int cls, const PanelDev &P, const TgtDev *tg, const uint32_t *d_n,
                           uint32_t nmax, uint32_t max_ww, uint32_t ncu, hipStream_t s);
hipError_t launch_plan(TgtDev *tg, BatchDev *B, const PlanArgs &A, hipStream_t s);
hipError_t launch_digest_count0_dev(const TgtDev *tg, const uint32_t *d_n, uint32_t nmax,
                                    hipStream_t s);
size_t cref_lds_bytes(const PanelDev &P, uint32_t maxK);
hipError_t cref_persist_prepare(const PanelDev &P, uint32_t maxK, int *occ);
bool cref_ident_ok(const PanelDev &P);
// site rows [m0, m0 + nsites) as 16-row blocks (panel PBWT)
hipError_t launch_site_blocks(const PanelDev &P, uint64_t m0, uint32_t nsites, uint16_t *blocks,
                              hipStream_t s);
hipError_t launch_cref_persist(const PanelDev &P, const TgtDev *tg, BatchDev *B,
                               const uint32_t *blockpref, const uint32_t *blockpref_id,
                               uint32_t maxK, const uint32_t *grid, hipStream_t s);

}  // namespace eimp
