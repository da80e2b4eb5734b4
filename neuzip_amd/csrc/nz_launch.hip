// The kernels of ONE precision (compile with -DNZ_S=7, 3, 1 or 0) and their
// host-side launchers; see nz_launch.h.
#ifndef NZ_S
#error "compile with -DNZ_S=<kept mantissa bits>"
#endif
#define NZ_TEMPLATES_ONLY
#include "nz_launch.h"

template <int S>
hipError_t nz_allow_encode_lds() {
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&nz_encode_kernel<S, 8>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, 96 * 1024);
  if (e == hipSuccess)
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(&nz_encode_kernel<S, 16>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, 96 * 1024);
  if (e == hipSuccess)
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(&nz_encode_kernel<S, 32>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, 96 * 1024);
  if (e == hipSuccess)
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(&nz_encode_kernel<S, 36>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, 96 * 1024);
  return e;
}

template <int S>
void nz_launch_encode(const NzEncBatch& b, int cls, dim3 grid, dim3 block, uint32_t lds, hipStream_t st) {
  switch (cls) {
    case 0: hipLaunchKernelGGL((nz_encode_kernel<S, 8>), grid, block, lds, st, b); break;
    case 1: hipLaunchKernelGGL((nz_encode_kernel<S, 16>), grid, block, lds, st, b); break;
    case 2: hipLaunchKernelGGL((nz_encode_kernel<S, 32>), grid, block, lds, st, b); break;
    case 3: hipLaunchKernelGGL((nz_encode_kernel<S, 36>), grid, block, lds, st, b); break;
    default: hipLaunchKernelGGL((nz_encode_long_kernel<S>), grid, dim3(NZ_ENC_LONG_THREADS), lds, st, b); break;
  }
}

template <int S>
void nz_launch_decode(const NzGeom& g, const void* comp, uint64_t comp_bytes, const void* packed, void* out,
                      uint32_t* d_status, const NzNorm& nm, uint32_t stream_out, hipStream_t st) {
  const bool one = nz_one_read(g.n_chunks, nz_compute_units(), stream_out);
  const uint32_t parts = nz_parts(g.n_chunks, g.spc, nz_compute_units(), stream_out);
  const size_t lds = NZ_DEC_LDS_BYTES(nz_part_rings(g.spc, parts), one);
  const dim3 gd((uint32_t)g.n_chunks * parts), bd(64 * g.spc);
#define NZ_DEC_LAUNCH(NORM, STREAM, ONE)                                                                       \
  hipLaunchKernelGGL((nz_decode_kernel<S, NORM, STREAM, ONE>), gd, bd, lds, st, (const uint8_t*)comp, comp_bytes, \
                     (const uint8_t*)packed, (uint16_t*)out, g, d_status, nm, parts)
  if (nm.bytes) {
    if (stream_out) NZ_DEC_LAUNCH(true, true, false);
    else if (one) NZ_DEC_LAUNCH(true, false, true);
    else NZ_DEC_LAUNCH(true, false, false);
  } else {
    if (stream_out) NZ_DEC_LAUNCH(false, true, false);
    else if (one) NZ_DEC_LAUNCH(false, false, true);
    else NZ_DEC_LAUNCH(false, false, false);
  }
#undef NZ_DEC_LAUNCH
}

template <int S>
void nz_launch_decode_batch(NzBatch& b, uint32_t grid, uint32_t max_spc, bool stream_out, uint32_t* d_status,
                            hipStream_t st) {
  const bool one = nz_one_read(grid, nz_compute_units(), stream_out);
  b.parts = nz_parts(grid, max_spc, nz_compute_units(), stream_out);
  const size_t lds = NZ_DEC_LDS_BYTES(nz_part_rings(max_spc, b.parts), one);
  const dim3 gd(grid * b.parts), bd(64 * max_spc);
#define NZ_BATCH_LAUNCH(NORM, STREAM, ONE) \
  hipLaunchKernelGGL((nz_decode_batch_kernel<S, NORM, STREAM, ONE>), gd, bd, lds, st, b, d_status)
  if (b.item[0].norm) {
    if (stream_out) NZ_BATCH_LAUNCH(true, true, false);
    else if (one) NZ_BATCH_LAUNCH(true, false, true);
    else NZ_BATCH_LAUNCH(true, false, false);
  } else {
    if (stream_out) NZ_BATCH_LAUNCH(false, true, false);
    else if (one) NZ_BATCH_LAUNCH(false, false, true);
    else NZ_BATCH_LAUNCH(false, false, false);
  }
#undef NZ_BATCH_LAUNCH
}

template <int S, bool ONE, bool WHOLE>
void nz_launch_gemv_form(const NzBatch& b, uint32_t grid, uint32_t max_spc, uint32_t* d_status, hipStream_t st) {
  const size_t lds = WHOLE && b.parts == 1 ? NZ_GEMV_LDS_BYTES(max_spc, ONE, b.x_rows)
                                           : NZ_DEC_LDS_BYTES(nz_part_rings(max_spc, b.parts), ONE);
  const dim3 gd(grid * b.parts), bd(64 * max_spc);
#define NZ_GEMV_LAUNCH(NORM, MR) \
  hipLaunchKernelGGL((nz_decode_gemv_kernel<S, NORM, MR, ONE, WHOLE>), gd, bd, lds, st, b, d_status)
  // a kernel for every number of activation rows
  if (b.item[0].norm) NZ_GEMV_LAUNCH(true, 1);  // (tensors with normalizers: one row only, the caller has checked)
  else switch (b.x_rows) {
    case 1: NZ_GEMV_LAUNCH(false, 1); break;
    case 2: NZ_GEMV_LAUNCH(false, 2); break;
    case 3: NZ_GEMV_LAUNCH(false, 3); break;
    case 4: NZ_GEMV_LAUNCH(false, 4); break;
    case 5: NZ_GEMV_LAUNCH(false, 5); break;
    case 6: NZ_GEMV_LAUNCH(false, 6); break;
    case 7: NZ_GEMV_LAUNCH(false, 7); break;
    default: NZ_GEMV_LAUNCH(false, 8); break;
  }
#undef NZ_GEMV_LAUNCH
}

template <int S>
void nz_launch_gemv(NzBatch& b, uint32_t grid, uint32_t max_spc, uint32_t* d_status, hipStream_t st) {
  b.parts = nz_parts(grid, max_spc, nz_compute_units(), false);
  const bool one = nz_one_read(grid, nz_compute_units(), false);
  if (b.in_features % NZ_GROUP_SYMS == 0) {
    if (one) nz_launch_gemv_form<S, true, true>(b, grid, max_spc, d_status, st);
    else nz_launch_gemv_form<S, false, true>(b, grid, max_spc, d_status, st);
  } else {
    if (one) nz_launch_gemv_form<S, true, false>(b, grid, max_spc, d_status, st);
    else nz_launch_gemv_form<S, false, false>(b, grid, max_spc, d_status, st);
  }
}

template <int S>
void nz_launch_rows(const NzGeom& g, const void* comp, uint64_t comp_bytes, const void* packed, uint16_t* out,
                    uint32_t* d_status, const NzNorm& nm, const long long* idx, uint32_t count, uint32_t row_len,
                    uint32_t cpr, hipStream_t st) {
  // segments of a chunk that a row can touch (one more where the chunk's last is a short one), and the table's record
  const bool aligned = g.seg_syms % row_len == 0 && g.chunk_syms % g.seg_syms == 0;
  const uint64_t touched = aligned ? 1u : ((uint64_t)row_len + g.seg_syms - 2) / g.seg_syms + 2;
  const bool one = nz_one_read((uint64_t)count * cpr, nz_compute_units(), false);
  const size_t lds = NZ_DEC_LDS_BYTES(touched + 1 < g.spc ? (uint32_t)touched + 1 : g.spc, one);
  const dim3 gd(count * cpr), bd(64 * g.spc);
#define NZ_ROWS_LAUNCH(NORM, WIDE)                                                                               \
  hipLaunchKernelGGL((nz_decode_rows_kernel<S, NORM, WIDE>), gd, bd, lds, st, (const uint8_t*)comp, comp_bytes, \
                     (const uint8_t*)packed, out, g, d_status, nm, idx, row_len, cpr)
  if (nm.bytes) {
    if (one) NZ_ROWS_LAUNCH(true, true);
    else NZ_ROWS_LAUNCH(true, false);
  } else {
    if (one) NZ_ROWS_LAUNCH(false, true);
    else NZ_ROWS_LAUNCH(false, false);
  }
#undef NZ_ROWS_LAUNCH
}

// NZ_PART (optional) cuts the unit into parts that a build can compile side by side:
// 0 = the encode kernels, 1 = decode, batch decode and row gather, 2 = the fused products,
// 12 = both of the latter; undefined = everything.  (Every part parses all of the kernels'
// source again: on eight cores two parts per precision build fastest, 68 s against 80 s
// with three and 91 s with one.)
#if !defined(NZ_PART) || NZ_PART == 0
template hipError_t nz_allow_encode_lds<NZ_S>();
template void nz_launch_encode<NZ_S>(const NzEncBatch&, int, dim3, dim3, uint32_t, hipStream_t);
#endif
#if !defined(NZ_PART) || NZ_PART == 1 || NZ_PART == 12
template void nz_launch_decode<NZ_S>(const NzGeom&, const void*, uint64_t, const void*, void*, uint32_t*, const NzNorm&,
                                     uint32_t, hipStream_t);
template void nz_launch_decode_batch<NZ_S>(NzBatch&, uint32_t, uint32_t, bool, uint32_t*, hipStream_t);
#endif
#if !defined(NZ_PART) || NZ_PART == 2 || NZ_PART == 12
template void nz_launch_gemv<NZ_S>(NzBatch&, uint32_t, uint32_t, uint32_t*, hipStream_t);
#endif
#if !defined(NZ_PART) || NZ_PART == 1 || NZ_PART == 12
template void nz_launch_rows<NZ_S>(const NzGeom&, const void*, uint64_t, const void*, uint16_t*, uint32_t*,
                                   const NzNorm&, const long long*, uint32_t, uint32_t, uint32_t, hipStream_t);
#endif

#if defined(NZ_PROBE_PHASES) && NZ_S == 7 && (!defined(NZ_PART) || NZ_PART == 0)
// measurement build only: cycles spent per phase of nz_encode_kernel<7, *>, summed over workgroups
extern "C" int nz_probe_read(unsigned long long* out, int reset) {
  if (hipMemcpyFromSymbol(out, HIP_SYMBOL(nz_probe_acc), sizeof(unsigned long long) * 8) != hipSuccess) return 1;
  if (reset) {
    unsigned long long z[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    if (hipMemcpyToSymbol(HIP_SYMBOL(nz_probe_acc), z, sizeof(z)) != hipSuccess) return 1;
  }
  return 0;
}
#endif
