// Contraction planner: loop IR -> one kernel launch.
//
// Replaces the reference's loop-nest lowering and primitive choice
//   BinaryContractionTpp::compile        reference src/backend/BinaryContractionTpp.cpp:4-127
//   ContractionOptimizer::optimize       reference src/basic/binary/ContractionOptimizer.cpp:47-74
//     (sort_and_fuse_iters :76-111, set_primitive_iters :232-584,
//      reorder_and_parallelize_iters :586-679)
//   ContractionBackend::set_kernel_shape reference src/basic/binary/ContractionBackend.cpp:518-678
//
// The reference picks a libxsmm GEMM/BRGEMM over the innermost unit-stride
// loops and runs every other loop on the host.  Here all loops of one type are
// flattened into a single kernel index (C -> grid batch, M -> MFMA rows,
// N -> MFMA columns, K -> reduction) and described by offset tables, so the
// whole contraction is one launch:
//   1. size-1 loops are dropped (ContractionOptimizer::remove_empty_iters, :113-121);
//   2. the kernel's column index (lanes 0..31 of a wave) is put on the
//      output's unit-stride type, swapping the roles of left and right when
//      the output is M-contiguous, so that epilogue stores coalesce;
//   3. inside each type the loops are ordered so that the operand's
//      unit-stride loop is innermost (the analogue of choosing the
//      primitive's unit-stride m/k loops); kernel rows the A operand is not
//      contiguous along follow the output's order instead;
//   4. the tables are enumerated and inspected: runs of consecutive offsets
//      select 16-byte vector loads along M/N or along K; a single-loop K index
//      becomes an affine offset (no table reads in the K loop);
//   5. the tile shape is chosen from dtype and the number of output tiles.
#include "etir_internal.h"
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <limits>
#include <sstream>

namespace etir {

int launch_contract_tile( int32_t tile, int32_t ma, int32_t mb, bool kaff, ContractArgs const & a,
                          uint32_t grid, hipStream_t stream );
int launch_contract_f64_64x64( int32_t ma, int32_t mb, bool kaff, ContractArgs const & a,
                               uint32_t grid, hipStream_t stream );
int launch_contract_cpx( bool f64, int32_t ma, int32_t mb, bool kaff, ContractArgs const & a,
                         uint32_t grid, hipStream_t stream );
int launch_contract_bf16_dma( int32_t ma, int32_t mb, int32_t variant, ContractArgs const & a,
                              uint32_t grid, hipStream_t stream );
int launch_contract_panel( ContractArgs const & a, hipStream_t stream );
int launch_contract_kwave( int32_t waves, int32_t kw, ContractArgs const & a, uint32_t grid,
                           hipStream_t stream );
int launch_contract_f32_dma( int32_t ma, int32_t mb, ContractArgs const & a, uint32_t grid, hipStream_t stream );
int launch_contract_f64_dma( ContractArgs const & a, uint32_t grid, hipStream_t stream );
int launch_contract_gemv( bool bf16_in, ContractArgs const & a, hipStream_t stream );
int launch_contract_skinny( bool bf16_in, ContractArgs const & a, hipStream_t stream );

namespace {

// tensor slots inside a loop
enum { T_L = 0, T_R = 1, T_AUX = 2, T_OUT = 3 };

struct Loop {
  int32_t type;
  int64_t size;
  int64_t s[4];
};

// enumerates sum_d digit_d * stride_d over the mixed-radix index of dims
// (outer -> inner)
std::vector< int64_t > enumerate( std::vector< Loop > const & dims, int slot ) {
  int64_t l_total = 1;
  for( Loop const & l_d : dims ) l_total *= l_d.size;
  std::vector< int64_t > l_tab( (std::size_t) l_total, 0 );
  if( l_total == 0 ) return l_tab;
  // fill from the innermost dim outwards: after processing a dim the first
  // l_filled entries hold the offsets of all inner digits
  int64_t l_filled = 1;
  for( int64_t l_di = (int64_t) dims.size() - 1; l_di >= 0; l_di-- ) {
    int64_t const l_sz = dims[l_di].size;
    int64_t const l_st = dims[l_di].s[slot];
    for( int64_t l_it = 1; l_it < l_sz; l_it++ ) {
      for( int64_t l_e = 0; l_e < l_filled; l_e++ ) {
        l_tab[l_it * l_filled + l_e] = l_tab[l_e] + l_it * l_st;
      }
    }
    l_filled *= l_sz;
  }
  return l_tab;
}

// true if tab is made of aligned runs of length v with unit increments and
// every run starts at a multiple of align
bool runs_contiguous( std::vector< int64_t > const & tab, int64_t v, int64_t align ) {
  if( (int64_t) tab.size() % v != 0 ) return false;
  for( std::size_t l_g = 0; l_g < tab.size(); l_g += v ) {
    if( tab[l_g] % align != 0 ) return false;
    for( int64_t l_e = 1; l_e < v; l_e++ ) {
      if( tab[l_g + l_e] != tab[l_g] + l_e ) return false;
    }
  }
  return true;
}

bool all_multiple( std::vector< int64_t > const & tab, int64_t align ) {
  for( int64_t l_v : tab ) if( l_v % align != 0 ) return false;
  return true;
}

bool fits_i32( std::vector< int64_t > const & tab ) {
  for( int64_t l_v : tab ) {
    if( l_v < 0 || l_v > std::numeric_limits< int32_t >::max() ) return false;
  }
  return true;
}

// sorts dims by their stride in `slot`, largest stride (outermost) first
void order_dims( std::vector< Loop > & dims, int slot ) {
  std::stable_sort( dims.begin(), dims.end(),
                    [slot]( Loop const & x, Loop const & y ) { return x.s[slot] > y.s[slot]; } );
}

// moves the first dim whose stride in `slot` is 1 to the innermost position;
// returns true if such a dim exists
bool unit_innermost( std::vector< Loop > & dims, int slot ) {
  for( std::size_t l_i = 0; l_i < dims.size(); l_i++ ) {
    if( dims[l_i].s[slot] == 1 ) {
      Loop l_d = dims[l_i];
      dims.erase( dims.begin() + l_i );
      dims.push_back( l_d );
      return true;
    }
  }
  return false;
}

std::string dims_str( std::vector< Loop > const & dims ) {
  std::ostringstream l_s;
  l_s << "[";
  for( std::size_t l_i = 0; l_i < dims.size(); l_i++ ) {
    if( l_i ) l_s << ",";
    l_s << dims[l_i].size;
  }
  l_s << "]";
  return l_s.str();
}

char const * mode_str( int32_t m ) {
  if( m == LOAD_VEC_MN ) return "vec_mn";
  if( m == LOAD_VEC_K )  return "vec_k";
  if( m == LOAD_VEC8_MN ) return "vec8_mn";
  if( m == LOAD_VEC8_K )  return "vec8_k";
  return "scalar";
}

char const * tile_str( int32_t t ) {
  switch( t ) {
    case TILE_F32_128x128:  return "f32_128x128x32";
    case TILE_F32_64x64:    return "f32_64x64x32";
    case TILE_BF16_256x256: return "bf16_256x256x64";
    case TILE_BF16_256x128: return "bf16_256x128x32";
    case TILE_BF16_DMA_256x256: return "bf16_dma_256x256";
    case TILE_BF16_DMA_256x128: return "bf16_dma_256x128";
    case TILE_BF16_DMA_128x128: return "bf16_dma_128x128";
    case TILE_BF16_128x128: return "bf16_128x128x64";
    case TILE_BF16_64x64:   return "bf16_64x64x64";
    case TILE_F64_64x64:    return "f64_64x64x16";
    case TILE_F64_DMA_128x128: return "f64_dma_128x128x16";
    case TILE_CPX_F32_64x64: return "cpx_f32_64x64x16";
    case TILE_CPX_F64_64x64: return "cpx_f64_64x64x16";
    case TILE_F32_KWAVE_32x32: return "f32_kwave_32x32";
    case TILE_F32_DMA_128x128: return "f32_dma_128x128x32";
    case TILE_GEMV:            return "gemv";
    case TILE_SKINNY:          return "skinny";
    case TILE_PANEL:           return "panel";
    default:                return "?";
  }
}

void tile_shape( int32_t t, int64_t & bm, int64_t & bn ) {
  switch( t ) {
    case TILE_F32_128x128:  bm = 128; bn = 128; break;
    case TILE_F32_64x64:    bm = 64;  bn = 64;  break;
    case TILE_BF16_256x256: bm = 256; bn = 256; break;
    case TILE_BF16_256x128: bm = 256; bn = 128; break;
    case TILE_BF16_DMA_256x256: bm = 256; bn = 256; break;
    case TILE_BF16_DMA_256x128: bm = 256; bn = 128; break;
    case TILE_F32_KWAVE_32x32: bm = 32; bn = 32; break;
    case TILE_BF16_128x128: bm = 128; bn = 128; break;
    case TILE_F32_DMA_128x128: bm = 128; bn = 128; break;
    case TILE_BF16_DMA_128x128: bm = 128; bn = 128; break;
    case TILE_F64_DMA_128x128: bm = 128; bn = 128; break;
    default:                bm = 64;  bn = 64;  break;
  }
}

}  // namespace

namespace {

// next 256-byte aligned piece of the caller's region, or a clear error
int place_take( DevicePlacement & place, std::size_t bytes, void ** out, char const * what ) {
  std::size_t const l_start = ( place.used + 255 ) & ~std::size_t( 255 );
  if( l_start + bytes > place.capacity ) {
    return fail( ETIR_UNDEFINED_ERROR, std::string( "contraction: the " ) + what + " need "
                                        + std::to_string( l_start + bytes ) + " bytes of scratch, more than the "
                                        + std::to_string( place.capacity ) + " the allocation-free entry point has" );
  }
  *out = place.base + l_start;
  place.used = l_start + bytes;
  return ETIR_SUCCESS;
}

int plan_contraction_impl( int64_t            num_loops,
                           int32_t const    * dim_types,
                           int64_t const    * sizes,
                           int64_t const    * strides_left,
                           int64_t const    * strides_right,
                           int64_t const    * strides_out_aux,
                           int64_t const    * strides_out,
                           int32_t            dtype_left,
                           int32_t            dtype_right,
                           int32_t            dtype_comp,
                           int32_t            dtype_out,
                           int32_t            ktype_first_touch,
                           int32_t            ktype_main,
                           int32_t            ktype_last_touch,
                           bool               allow_split,
                           ContractionPlan  & plan,
                           DevicePlacement  * place,
                           bool               dry = false,
                           bool               copied = false ) {
  // dry: tile, load modes and split (those of its partial contraction) only,
  // no device memory; copied: operands of a packed contraction
  plan = ContractionPlan();
  plan.placed = ( place != nullptr );

  // ---------------------------------------------------------------- checks
  bool const l_f32  = dtype_left == ETIR_FP32 && dtype_right == ETIR_FP32
                   && dtype_comp == ETIR_FP32 && dtype_out == ETIR_FP32;
  bool const l_bf16 = dtype_left == ETIR_BF16 && dtype_right == ETIR_BF16
                   && dtype_comp == ETIR_FP32
                   && ( dtype_out == ETIR_FP32 || dtype_out == ETIR_BF16 );
  bool const l_f64  = dtype_left == ETIR_FP64 && dtype_right == ETIR_FP64
                   && dtype_comp == ETIR_FP64 && dtype_out == ETIR_FP64;
  if( !l_f32 && !l_bf16 && !l_f64 ) {
    return fail( ETIR_INVALID_DTYPE, "contraction: unsupported dtype combination" );
  }
  // complex: CPX_MADD with the reference BLAS backend's touch kernels
  // (BinaryContractionBlas.cpp:68-80)
  bool const l_cpx = ( ktype_main == ETIR_KTYPE_CPX_MADD );
  if( l_cpx ) {
    if( l_bf16 ) return fail( ETIR_INVALID_DTYPE, "contraction: complex kernels take FP32 or FP64" );
    if(    ktype_first_touch != ETIR_KTYPE_ZERO && ktype_first_touch != ETIR_KTYPE_CPX_ZERO
        && ktype_first_touch != ETIR_KTYPE_UNDEFINED ) {
      return fail( ETIR_INVALID_KTYPE, "contraction: unsupported complex first-touch kernel" );
    }
    if( ktype_last_touch != ETIR_KTYPE_UNDEFINED ) {
      return fail( ETIR_INVALID_KTYPE, "contraction: complex contractions have no last-touch kernel" );
    }
  }
  else {
    if( ktype_main != ETIR_KTYPE_MADD ) {
      return fail( ETIR_INVALID_KTYPE, "contraction: main kernel must be MADD or CPX_MADD" );
    }
    if(    ktype_first_touch != ETIR_KTYPE_ZERO && ktype_first_touch != ETIR_KTYPE_COPY
        && ktype_first_touch != ETIR_KTYPE_ADD  && ktype_first_touch != ETIR_KTYPE_UNDEFINED ) {
      return fail( ETIR_COMPILATION_FAILED, "contraction: unsupported first-touch kernel" );
    }
    if(    ktype_last_touch != ETIR_KTYPE_RELU && ktype_last_touch != ETIR_KTYPE_ADD
        && ktype_last_touch != ETIR_KTYPE_UNDEFINED ) {
      return fail( ETIR_COMPILATION_FAILED, "contraction: unsupported last-touch kernel" );
    }
  }
  if( num_loops < 0 || ( num_loops > 0 && ( dim_types == nullptr || sizes == nullptr
                                            || strides_left == nullptr || strides_right == nullptr
                                            || strides_out == nullptr ) ) ) {
    return fail( ETIR_COMPILATION_FAILED, "contraction: invalid loop arrays" );
  }

  plan.dtype_in    = dtype_left;
  plan.dtype_comp  = dtype_comp;
  plan.dtype_out   = dtype_out;
  plan.first_touch = ktype_first_touch;
  plan.last_touch  = ktype_last_touch;
  plan.needs_aux   =    ktype_first_touch == ETIR_KTYPE_COPY
                     || ktype_first_touch == ETIR_KTYPE_ADD
                     || ktype_last_touch  == ETIR_KTYPE_ADD;
  // without explicit aux strides the aux tensor shares the output's layout
  // (reference src/backend/BinaryContractionTpp.cpp:36-41)
  int64_t const * l_s_aux = strides_out_aux != nullptr ? strides_out_aux : strides_out;

  // ------------------------------------------------------------- loop sets
  std::vector< Loop > l_c, l_m, l_n, l_k, l_x;
  for( int64_t l_lo = 0; l_lo < num_loops; l_lo++ ) {
    if( sizes[l_lo] < 0 ) return fail( ETIR_COMPILATION_FAILED, "contraction: negative loop size" );
    if(    strides_left[l_lo] < 0 || strides_right[l_lo] < 0 || strides_out[l_lo] < 0
        || l_s_aux[l_lo] < 0 ) {
      return fail( ETIR_COMPILATION_FAILED, "contraction: negative stride" );
    }
    Loop l_lp{ dim_types[l_lo], sizes[l_lo],
               { strides_left[l_lo], strides_right[l_lo], l_s_aux[l_lo], strides_out[l_lo] } };
    if( l_lp.type == ETIR_DIM_I || l_lp.type == ETIR_DIM_J ) continue;
    if( l_lp.type == ETIR_DIM_CPX ) {
      l_x.push_back( l_lp );
      continue;
    }
    if( l_lp.size == 1 ) continue;
    if(      l_lp.type == ETIR_DIM_C ) l_c.push_back( l_lp );
    else if( l_lp.type == ETIR_DIM_M ) l_m.push_back( l_lp );
    else if( l_lp.type == ETIR_DIM_N ) l_n.push_back( l_lp );
    else if( l_lp.type == ETIR_DIM_K ) l_k.push_back( l_lp );
    else return fail( ETIR_COMPILATION_FAILED, "contraction: invalid dimension type" );
  }

  if( l_cpx != ( l_x.size() > 0 ) ) {
    return fail( ETIR_INVALID_CPX_DIM, "contraction: CPX_MADD needs exactly one CPX loop and CPX loops need CPX_MADD" );
  }
  if( l_x.size() > 1 || ( l_cpx && l_x[0].size != 2 ) ) {
    return fail( ETIR_INVALID_CPX_DIM, "contraction: the complex loop must be unique and of size 2" );
  }
  auto prod = []( std::vector< Loop > const & d ) {
    int64_t l_p = 1;
    for( Loop const & l_x : d ) l_p *= l_x.size;
    return l_p;
  };
  int64_t const l_size_c = prod( l_c );
  int64_t const l_size_m = prod( l_m );
  int64_t const l_size_n = prod( l_n );
  int64_t const l_size_k = prod( l_k );

  // ------------------------------------------------------------ role swap
  // kernel columns (lane index) go to the output's unit-stride type
  bool l_swap = false;
  for( Loop const & l_x : l_m ) if( l_x.s[T_OUT] == 1 ) l_swap = true;
  plan.swapped = l_swap;

  // kernel operand slots: A (rows), B (columns)
  int const l_sa = l_swap ? T_R : T_L;
  int const l_sb = l_swap ? T_L : T_R;
  std::vector< Loop > l_km = l_swap ? l_n : l_m;   // kernel-M loops (A, aux, out)
  std::vector< Loop > l_kn = l_swap ? l_m : l_n;   // kernel-N loops (B, aux, out)
  int64_t const l_kern_m = l_swap ? l_size_n : l_size_m;
  int64_t const l_kern_n = l_swap ? l_size_m : l_size_n;

  int64_t const l_esz = ( dtype_left == ETIR_BF16 ) ? 2 : ( dtype_left == ETIR_FP64 ? 8 : 4 );
  int64_t const l_vk  = 16 / l_esz;   // elements per 16-byte vector

  // ordering: kernel rows follow A when A is read along them, otherwise the
  // output (neighbouring tile rows then sit close in memory for the stores)
  bool l_a_unit_m = false;
  for( Loop const & l_x : l_km ) if( l_x.s[l_sa] == 1 ) l_a_unit_m = true;
  order_dims( l_km, l_a_unit_m ? l_sa : T_OUT );
  if( l_a_unit_m ) unit_innermost( l_km, l_sa );
  order_dims( l_kn, T_OUT );
  if( !unit_innermost( l_kn, T_OUT ) ) unit_innermost( l_kn, l_sb );
  // K: the operand whose unit-stride loop is a K loop decides the order
  bool l_a_unit_k = false, l_b_unit_k = false;
  for( Loop const & l_x : l_k ) {
    if( l_x.s[l_sa] == 1 ) l_a_unit_k = true;
    if( l_x.s[l_sb] == 1 ) l_b_unit_k = true;
  }
  int const l_k_slot = l_a_unit_k ? l_sa : ( l_b_unit_k ? l_sb : l_sa );
  order_dims( l_k, l_k_slot );
  unit_innermost( l_k, l_k_slot );
  order_dims( l_c, T_OUT );

  // --------------------------------------------------------------- tables
  std::vector< int64_t > l_tc_a   = enumerate( l_c, l_sa );
  std::vector< int64_t > l_tc_b   = enumerate( l_c, l_sb );
  std::vector< int64_t > l_tc_aux = enumerate( l_c, T_AUX );
  std::vector< int64_t > l_tc_out = enumerate( l_c, T_OUT );
  std::vector< int64_t > l_tm_a   = enumerate( l_km, l_sa );
  std::vector< int64_t > l_tm_aux = enumerate( l_km, T_AUX );
  std::vector< int64_t > l_tm_out = enumerate( l_km, T_OUT );
  std::vector< int64_t > l_tn_b   = enumerate( l_kn, l_sb );
  std::vector< int64_t > l_tn_aux = enumerate( l_kn, T_AUX );
  std::vector< int64_t > l_tn_out = enumerate( l_kn, T_OUT );
  std::vector< int64_t > l_tk_a   = enumerate( l_k, l_sa );
  std::vector< int64_t > l_tk_b   = enumerate( l_k, l_sb );

  int64_t const l_max_i32 = std::numeric_limits< int32_t >::max();
  if(    l_size_m > l_max_i32 || l_size_n > l_max_i32 || l_size_k > l_max_i32
      || l_size_c > l_max_i32 ) {
    return fail( ETIR_COMPILATION_FAILED, "contraction: flattened index exceeds int32" );
  }
  if(    !fits_i32( l_tm_a ) || !fits_i32( l_tm_aux ) || !fits_i32( l_tm_out )
      || !fits_i32( l_tn_b ) || !fits_i32( l_tn_aux ) || !fits_i32( l_tn_out )
      || !fits_i32( l_tk_a ) || !fits_i32( l_tk_b ) ) {
    return fail( ETIR_COMPILATION_FAILED, "contraction: per-type offsets exceed int32" );
  }
  int64_t const l_total_entries = 4 * l_size_c + 3 * ( l_size_m + l_size_n ) + 2 * l_size_k;
  if( l_total_entries > ( int64_t( 1 ) << 27 ) ) {
    return fail( ETIR_COMPILATION_FAILED, "contraction: offset tables too large" );
  }

  // ------------------------------------------------------- load modes
  auto pick_mode = [&]( std::vector< int64_t > const & rows,
                        std::vector< int64_t > const & tk,
                        std::vector< int64_t > const & tc ) -> int32_t {
    // 16-byte vectors of consecutive rows (4 fp32 / 8 bf16)
    if(    rows.size() > 0 && runs_contiguous( rows, l_vk, l_vk )
        && all_multiple( tk, l_vk ) && all_multiple( tc, l_vk ) ) {
      return LOAD_VEC_MN;
    }
    // 16-byte vectors along K
    if(    tk.size() > 0 && runs_contiguous( tk, l_vk, l_vk )
        && all_multiple( rows, l_vk ) && all_multiple( tc, l_vk ) ) {
      return LOAD_VEC_K;
    }
    // fp32 runs of even length that are not multiples of 4 (odd mode sizes
    // times 2, as in the einsum_benchmark MERA network): 8-byte vectors on
    // the generic fp32 tiles
    if( l_f32 && !l_cpx ) {
      if(    rows.size() > 0 && runs_contiguous( rows, 2, 2 )
          && all_multiple( tk, 2 ) && all_multiple( tc, 2 ) ) {
        return LOAD_VEC8_MN;
      }
      if(    tk.size() > 0 && runs_contiguous( tk, 2, 2 )
          && all_multiple( rows, 2 ) && all_multiple( tc, 2 ) ) {
        return LOAD_VEC8_K;
      }
    }
    return LOAD_SCALAR;
  };
  plan.mode_a = pick_mode( l_tm_a, l_tk_a, l_tc_a );
  plan.mode_b = pick_mode( l_tn_b, l_tk_b, l_tc_b );
  // complex: the imaginary parts are loaded like the real ones from base +
  // cpx stride, so that offset has to keep the 16-byte vector alignment
  if( l_cpx && l_x[0].s[l_sa] % l_vk != 0 ) plan.mode_a = LOAD_SCALAR;
  if( l_cpx && l_x[0].s[l_sb] % l_vk != 0 ) plan.mode_b = LOAD_SCALAR;

  bool l_k_affine = true;
  int64_t l_sk_a = l_tk_a.size() > 1 ? l_tk_a[1] : 0;
  int64_t l_sk_b = l_tk_b.size() > 1 ? l_tk_b[1] : 0;
  for( std::size_t l_i = 0; l_i < l_tk_a.size(); l_i++ ) {
    if( l_tk_a[l_i] != int64_t( l_i ) * l_sk_a || l_tk_b[l_i] != int64_t( l_i ) * l_sk_b ) {
      l_k_affine = false;
      break;
    }
  }

  // ---------------------------------------------------------- tile choice
  auto n_tiles = [&]( int32_t t ) {
    int64_t l_bm, l_bn;
    tile_shape( t, l_bm, l_bn );
    return ( ( l_kern_m + l_bm - 1 ) / l_bm ) * ( ( l_kern_n + l_bn - 1 ) / l_bn ) * l_size_c;
  };
  int64_t const l_cus = 256;
  // useful fraction of the padded tile grid times the fraction of CUs with a
  // tile: M = 64 on 128 x 128 tiles wastes half of every tile
  auto score = [&]( int32_t t ) {
    int64_t l_bm, l_bn;
    tile_shape( t, l_bm, l_bn );
    double const l_pad = double( ( ( l_kern_m + l_bm - 1 ) / l_bm ) * l_bm )
                       * double( ( ( l_kern_n + l_bn - 1 ) / l_bn ) * l_bn );
    double const l_util = l_pad > 0.0 ? double( l_kern_m ) * double( l_kern_n ) / l_pad : 1.0;
    return l_util * std::min( 1.0, double( n_tiles( t ) ) / double( l_cus ) );
  };
  if( l_cpx ) {
    plan.tile = l_f64 ? TILE_CPX_F64_64x64 : TILE_CPX_F32_64x64;
  }
  else if( l_f64 ) {
    plan.tile = TILE_F64_64x64;
  }
  else if( l_f32 ) {
    // the larger tile unless the smaller one wastes clearly less
    plan.tile = ( score( TILE_F32_128x128 ) >= 0.95 * score( TILE_F32_64x64 ) ) ? TILE_F32_128x128 : TILE_F32_64x64;
  }
  else {
    if(      n_tiles( TILE_BF16_256x128 ) >= 2 * l_cus ) plan.tile = TILE_BF16_256x128;
    else if( n_tiles( TILE_BF16_128x128 ) >= l_cus ) plan.tile = TILE_BF16_128x128;
    else                                             plan.tile = TILE_BF16_64x64;
  }
  // bf16 direct-to-LDS kernels: 16-byte vector modes on both operands, affine
  // K, every byte offset below the buffer range (2^31)
  auto max_of = []( std::vector< int64_t > const & t ) {
    int64_t l_m = 0;
    for( int64_t l_v : t ) l_m = std::max( l_m, l_v );
    return l_m;
  };
  bool const l_dma_ok =
         l_bf16
      && ( plan.mode_a == LOAD_VEC_MN || plan.mode_a == LOAD_VEC_K )
      && ( plan.mode_b == LOAD_VEC_MN || plan.mode_b == LOAD_VEC_K )
      && l_k_affine
      && 2 * ( max_of( l_tm_a ) + std::max< int64_t >( l_size_k - 1, 0 ) * l_sk_a ) + 64 < ( int64_t( 1 ) << 31 )
      && 2 * ( max_of( l_tn_b ) + std::max< int64_t >( l_size_k - 1, 0 ) * l_sk_b ) + 64 < ( int64_t( 1 ) << 31 )
      && 2 * int64_t( 64 ) * std::max( l_sk_a, l_sk_b ) * ( ( l_size_k + 63 ) / 64 + 4 ) < ( int64_t( 1 ) << 31 );
  plan.tile_fallback = plan.tile;
  // fp64 direct-to-LDS kernel: both operands K-contiguous, byte offsets below
  // the buffer range (the loads of the step past the last one are issued
  // too), and fewer rounds of tiles: a round of one 128 x 128 tile per CU takes
  // as long as three of 64 x 64 ones (per unit of K 0.12 us, 0.04), also a last
  // one that is nearly empty.  mk,nk->mn, 64 / 128 tiles: 2544 x 1539 x 2442 (4
  // rounds, 2) 396 / 581 us, 3320 x 1491 x 574 (5, 2) 127 / 147, K = 98 with 9
  // and 3 rounds 56 / 61; 252 tiles, K = 1534 (4, 1) 253 / 207.  Up to a K of 64
  // loads and stores count, and the larger tiles only have to fill the chip (5
  // rounds and 2, K = 54: 27.8 / 27.6; 6 and 2, K = 38: 27.8 / 24.2); so they do
  // for copied operands (aecf,bfde->abcd 48,46,43,44,41,39, 272 tiles: 419 us
  // packed on them, 862 in place)
  auto rounds = [&]( int32_t t ) { return ( n_tiles( t ) + l_cus - 1 ) / l_cus; };
  if(    l_f64 && !l_cpx && plan.mode_a == LOAD_VEC_K && plan.mode_b == LOAD_VEC_K && l_k_affine && l_sk_a == 1
      && l_sk_b == 1 && 8 * ( std::max( max_of( l_tm_a ), max_of( l_tn_b ) ) + l_size_k + 64 ) < ( int64_t( 1 ) << 31 )
      && (    3 * rounds( TILE_F64_DMA_128x128 ) < rounds( TILE_F64_64x64 )
           || ( ( copied || l_size_k <= 64 ) && score( TILE_F64_DMA_128x128 ) >= 0.9 * score( TILE_F64_64x64 ) ) ) ) {
    plan.tile = TILE_F64_DMA_128x128;
  }
  // 256 x 256 tiles where their persistent scheduled loop runs (both operands
  // row-contiguous, whole tiles, plain fp32 output in 32-column runs: 4096 a
  // side 109 us) and, with row-contiguous operands, where its one-tile form
  // walks a long K and leaves no large part of the last round of CUs idle
  // (km,kn->mn, 256 against 128 tiles: 4072 x 4072 x 8192 230 / 314 us, 8184 x
  // 4088 x 8192 463 / 595, x 4096 279 / 315; but 4072 x 4072 x 4096 142 / 144, x
  // 2048 100 / 84, and 2552 x 8184 x 8192, 320 tiles, 422 / 411).  Everything
  // else with a 128 x 128 tile per CU takes those, two workgroups per CU,
  // against the generic 256 x 256 loop (one) and the register-staged tiles:
  // mk,nk->mn 4096 a side 168 -> 126 us, 8192 x 1024 x 4096 82 -> 66 us, 4072 x
  // 2048 x 2048 44 -> 38 us, 2304 x 2304 x 1024 20 -> 18 us; bf16 results
  // (16-byte stores) 55 -> 36 us at 4072 x 2048 x 2048
  std::size_t l_run_n = 1;
  while( l_run_n < l_tn_out.size() && l_tn_out[l_run_n] == l_tn_out[l_run_n - 1] + 1 ) l_run_n++;
  // persistent_dma_eligible, before the kernel's arguments exist
  bool const l_persistent =
         plan.mode_a == LOAD_VEC_MN && plan.mode_b == LOAD_VEC_MN && dtype_out == ETIR_FP32
      && ktype_first_touch == ETIR_KTYPE_ZERO && ktype_last_touch == ETIR_KTYPE_UNDEFINED
      && l_kern_m % 256 == 0 && l_kern_n % 256 == 0 && l_run_n >= 32
      && ( l_run_n % 32 == 0 || l_run_n == l_tn_out.size() )
      && 4 * ( max_of( l_tm_out ) + max_of( l_tn_out ) ) + 4 < ( int64_t( 1 ) << 32 );
  plan.scattered = l_run_n < 32 && l_run_n < l_tn_out.size() && l_tm_out.size() > 1
                && l_tm_out[1] != l_tm_out[0] + int64_t( l_run_n );
  int64_t const l_t256 = n_tiles( TILE_BF16_DMA_256x256 );
  double const l_last = double( l_t256 ) / double( ( l_t256 + l_cus - 1 ) / l_cus * l_cus + ( l_t256 == 0 ) );
  bool const l_long_k = plan.mode_a == LOAD_VEC_MN && plan.mode_b == LOAD_VEC_MN
                     && (    ( l_size_k >= 8192 && l_last >= 0.75 )
                          || ( l_size_k >= 4096 && l_last >= 0.95 && l_t256 >= 2 * l_cus ) );
  if( l_dma_ok && ( l_persistent || l_long_k ) && l_t256 >= l_cus ) plan.tile = TILE_BF16_DMA_256x256;
  else if( l_dma_ok && n_tiles( TILE_BF16_DMA_128x128 ) >= l_cus ) plan.tile = TILE_BF16_DMA_128x128;
  // the fp32 direct-to-LDS kernel: where the planner chose the 128 x 128 fp32
  // tile, under the same conditions (4-byte elements; the loads of the step
  // past the last one are issued too); a K that is not affine up to 1024,
  // whose offset tables the kernel copies into LDS
  int64_t const l_bytes_max = int64_t( 1 ) << 31;
  bool const l_f32_dma_k =
         ( l_k_affine
           && 4 * ( max_of( l_tm_a ) + std::max< int64_t >( l_size_k - 1, 0 ) * l_sk_a ) + 64 < l_bytes_max
           && 4 * ( max_of( l_tn_b ) + std::max< int64_t >( l_size_k - 1, 0 ) * l_sk_b ) + 64 < l_bytes_max
           && 4 * int64_t( 32 ) * std::max( l_sk_a, l_sk_b ) * ( ( l_size_k + 31 ) / 32 + 2 ) < l_bytes_max )
      || ( !l_k_affine && l_size_k <= 1024
           && 4 * ( max_of( l_tm_a ) + max_of( l_tk_a ) ) + 64 < l_bytes_max
           && 4 * ( max_of( l_tn_b ) + max_of( l_tk_b ) ) + 64 < l_bytes_max );
  bool const l_f32_dma_ok =
         l_f32 && !l_cpx
      && ( plan.mode_a == LOAD_VEC_MN || plan.mode_a == LOAD_VEC_K )
      && ( plan.mode_b == LOAD_VEC_MN || plan.mode_b == LOAD_VEC_K )
      && l_f32_dma_k;
  if( l_f32_dma_ok && plan.tile == TILE_F32_128x128 ) plan.tile = TILE_F32_DMA_128x128;
  if( char const * l_env = ( l_f64 || l_cpx ) ? nullptr : std::getenv( "ETIR_TILE" ) ) {
    // diagnostic override of the tile heuristic (must match the dtype)
    int32_t l_t = std::atoi( l_env );
    bool const l_t_f32 = ( l_t == TILE_F32_128x128 || l_t == TILE_F32_64x64
                           || ( l_t == TILE_F32_DMA_128x128 && l_f32_dma_ok ) );
    bool const l_t_dma = ( l_t == TILE_BF16_DMA_256x256 || l_t == TILE_BF16_DMA_256x128 );
    bool const l_t_ok = ( ( ( l_t >= 0 && l_t <= TILE_BF16_DMA_256x128 ) || l_t == TILE_F32_DMA_128x128 )
                          && l_t != TILE_F64_64x64 && l_t_f32 == l_f32 )
                     && ( !l_t_dma || l_dma_ok )
                     && ( l_t != TILE_BF16_DMA_256x128
                          || ( plan.mode_a == LOAD_VEC_MN && plan.mode_b == LOAD_VEC_MN ) );
    if( l_t_ok ) plan.tile = l_t;
  }
  // VEC_MN x VEC_MN runs the explicitly scheduled BK 32 / 4-stage main loop;
  // the other pairings (VEC_K needs 64-wide k rows; under ETIR_TILE) the generic BK 64 / 2-stage one
  // (3: the persistent variant of the scheduled loop, for contractions it
  // runs -- all tiles full, plain fp32 stores -- decided at launch)
  plan.dma_variant = ( plan.mode_a == LOAD_VEC_MN && plan.mode_b == LOAD_VEC_MN ) ? 3 : 0;
  if( char const * l_env = std::getenv( "ETIR_DMA_VARIANT" ) ) {
    // diagnostic override, only values whose kernel runs on this plan's
    // 256 x 256 tile grid: 0 forces the generic BK 64 / 2-stage loop, 1 the
    // one-tile scheduled loop and 3 its persistent form (both VEC_MN x
    // VEC_MN only); anything else is ignored (the 256 x 128 kernel has a
    // tile grid of its own and is chosen by ETIR_TILE)
    int32_t const l_v = std::atoi( l_env );
    if( l_v == 0 ) plan.dma_variant = 0;
    if( ( l_v == 1 || l_v == 3 ) && plan.dma_variant == 3 ) plan.dma_variant = l_v;
  }

  // ------------------------------------------------------- matrix-vector
  // One free side of extent 1 pads every MFMA tile to one row in 64: one
  // thread per output element instead, when the long side's operand is
  // unit-stride along it (coalesced loads), K is short enough for a
  // per-thread loop and the outputs fill the chip (256 CUs x 1024 threads).
  // ETIR_TILE=13 forces it for any M == 1 or N == 1 shape.
  {
    bool const l_mv_shape = ( l_f32 || l_bf16 ) && !l_cpx && ( l_kern_m == 1 || l_kern_n == 1 );
    char const * l_env_t = std::getenv( "ETIR_TILE" );
    bool const l_forced = l_mv_shape && l_env_t != nullptr && std::atoi( l_env_t ) == TILE_GEMV;
    bool const l_long_vec = ( l_kern_m == 1 && l_kern_n > 1 ) ? ( plan.mode_b == LOAD_VEC_MN )
                          : ( l_kern_n == 1 && l_kern_m > 1 ) ? ( plan.mode_a == LOAD_VEC_MN ) : false;
    bool const l_mv_ok = l_mv_shape && l_long_vec && l_size_k <= 256
                      && l_size_c * l_kern_m * l_kern_n >= 1024 * l_cus
                      && l_env_t == nullptr && std::getenv( "ETIR_NO_GEMV" ) == nullptr;
    if( l_mv_ok || l_forced ) plan.tile = TILE_GEMV;
  }

  // ------------------------------------------------- one short free side
  // A free side of 2 to 64 pads most of every MFMA tile, and with a short K
  // the tiles are bound by their load round trip and stores: one thread per
  // index of the long side instead, the short side's outputs in registers
  // (einsum_benchmark MERA, M = 11, N = 415800, K = 24: 28 us on 64 x 64
  // tiles).  Where the short side is 17-64, only with K <= 64 (the FMAs per
  // long-operand byte grow with the short side); at least 256 workgroups of
  // 256 threads.  ETIR_TILE=14 forces it for any short side of 2 to 64.
  {
    int64_t const l_sh = std::min( l_kern_m, l_kern_n );
    int64_t const l_lo = std::max( l_kern_m, l_kern_n );
    bool const l_sk_shape = ( l_f32 || l_bf16 ) && !l_cpx && plan.tile != TILE_GEMV && l_sh >= 2 && l_sh <= 64
                         && l_size_c <= 65535;
    char const * l_env_t = std::getenv( "ETIR_TILE" );
    bool const l_forced = l_sk_shape && l_env_t != nullptr && std::atoi( l_env_t ) == TILE_SKINNY;
    // not where the output's unit-stride dim is a C dim: a thread's stores
    // would then be C elements apart (TCCG efbadx,cfx->abcdex: 2.3 against
    // 7.8 TFLOP/s on the tiles, which walk C fastest there)
    int64_t l_os_c = std::numeric_limits< int64_t >::max();
    int64_t l_os_mn = std::numeric_limits< int64_t >::max();
    for( Loop const & l_x : l_c ) if( l_x.size > 1 ) l_os_c = std::min( l_os_c, l_x.s[T_OUT] );
    for( auto const * l_set : { &l_m, &l_n } ) {
      for( Loop const & l_x : *l_set ) if( l_x.size > 1 ) l_os_mn = std::min( l_os_mn, l_x.s[T_OUT] );
    }
    bool const l_sk_ok = l_sk_shape && ( l_sh <= 16 || l_size_k <= 64 ) && l_os_mn < l_os_c
                      && l_size_c * ( ( l_lo + 255 ) / 256 ) >= l_cus && l_env_t == nullptr
                      && std::getenv( "ETIR_NO_SKINNY" ) == nullptr;
    if( l_sk_ok || l_forced ) plan.tile = TILE_SKINNY;
  }

  // ------------------------------------- short K, one free side of 65-256
  // With K <= 64 an MFMA tile lives for one load round trip and its stores
  // (einsum_benchmark MERA root, M = 177147, N = 243, K = 50: 73 us on 128 x
  // 128 tiles, 62 here): the short operand stays in LDS for the whole launch
  // and persistent workgroups stream panels of the long side, each panel's
  // stores issued between the next one's MFMAs.  fp32, no C dims, first
  // touch ZERO, last touch none or RELU, the long operand affine along its
  // side, at least four panels per CU (each workgroup pays about one panel
  // of set-up: M = 16384 k x 243 x 50 at 2 / 4 panels per CU 22.7 / 32.1 us
  // against 21.1 / 40.9 on the tiles).  ETIR_TILE=15 forces it where the
  // shape allows (a long side of at least one panel), ETIR_NO_PANEL turns it
  // off.
  {
    int64_t const l_sh = std::min( l_kern_m, l_kern_n );
    int64_t const l_lo = std::max( l_kern_m, l_kern_n );
    bool const l_res_a = l_kern_m <= l_kern_n;
    std::vector< int64_t > const & l_tl = l_res_a ? l_tn_b : l_tm_a;
    bool l_aff = true;
    int64_t const l_st = l_tl.size() > 1 ? l_tl[1] : 0;
    for( std::size_t l_i = 0; l_i < l_tl.size() && l_aff; l_i++ ) l_aff = ( l_tl[l_i] == int64_t( l_i ) * l_st );
    l_aff = l_aff && l_st >= 0 && l_st <= std::numeric_limits< int32_t >::max();
    int64_t l_mo = 0, l_no = 0;
    for( int64_t l_v : l_tm_out ) l_mo = std::max( l_mo, l_v );
    for( int64_t l_v : l_tn_out ) l_no = std::max( l_no, l_v );
    bool const l_pn_shape = l_f32 && !l_cpx && plan.tile != TILE_GEMV && plan.tile != TILE_SKINNY
                         && l_size_c == 1 && l_sh > 64 && l_sh <= 256 && l_size_k >= 1 && l_size_k <= 64
                         && ktype_first_touch == ETIR_KTYPE_ZERO
                         && ( ktype_last_touch == ETIR_KTYPE_UNDEFINED || ktype_last_touch == ETIR_KTYPE_RELU )
                         && !plan.needs_aux && l_aff && 4 * ( l_mo + l_no + 1 ) <= int64_t( 0xffffff00u );
    int64_t const l_pl = ( l_sh > 128 ) ? 64 : 128;
    char const * l_env_t = std::getenv( "ETIR_TILE" );
    bool const l_forced = l_pn_shape && l_lo >= l_pl && l_env_t != nullptr && std::atoi( l_env_t ) == TILE_PANEL;
    bool const l_pn_ok = l_pn_shape && ( l_lo + l_pl - 1 ) / l_pl >= 4 * l_cus && l_env_t == nullptr
                      && std::getenv( "ETIR_NO_PANEL" ) == nullptr;
    if( l_pn_ok || l_forced ) plan.tile = TILE_PANEL;
  }

  // ------------------------------------------- long K on few large tiles
  // The 64 x 64 tile fills the chip where fewer than 256 of the 128 x 128
  // tiles exist, but runs at about half the fp32 direct-to-LDS kernel's rate;
  // with K >= 2048 the larger tile split over K (below) is faster (1024 x 1024
  // x 8192: 148 us against 198; 1215 x 924 x 4620: 139 against 188).  Undone
  // after the split block if K does not split.
  int32_t const l_tile_unsplit = plan.tile;
  bool const l_big_k_split = allow_split && l_f32_dma_ok && plan.tile == TILE_F32_64x64 && l_size_k >= 2048
                          && n_tiles( TILE_F32_128x128 ) < l_cus && std::getenv( "ETIR_TILE" ) == nullptr;
  if( l_big_k_split ) plan.tile = TILE_F32_DMA_128x128;

  int64_t l_bm, l_bn;
  tile_shape( plan.tile, l_bm, l_bn );

  // --------------------------------------------- K split inside a workgroup
  // Few output tiles, both operands K-contiguous fp32, K up to 4096: 32 x 32
  // tiles (4x the workgroups of 64 x 64) with K divided over the 16 waves of
  // each workgroup, whose partial tiles are added in LDS -- one launch, no
  // workspace (the alternative below, split K, sends S partial outputs
  // through memory to a second kernel).  At most 512 of them, one round of
  // two workgroups per CU (bench_mlp's 576-tile nodes: 95 us/eval with them,
  // 90 on split K).  Fewer than 128 only up to K = 512: 128 x 128 x 256 takes
  // 5.1 us against 8.4 on 64 x 64 tiles, whose four workgroups walk K step by
  // step (K = 96: 3.9 against 4.8; 512: 7.3 against 8.8 split); from 768 on
  // split K has more workgroups (K = 1024: 11.7 against 9.1).  Up to K = 96
  // only one round of one workgroup per CU (256 tiles, 512 x 512: 4.2 us
  // against 5.1; 484 tiles, 704 x 704: 5.6 against 5.3; K = 112: 5.6 against 5.8)
  {
    int64_t const l_t32 = n_tiles( TILE_F32_KWAVE_32x32 );
    bool const l_kw_ok = l_f32 && plan.tile != TILE_GEMV && plan.tile != TILE_SKINNY && plan.tile != TILE_PANEL && plan.mode_a == LOAD_VEC_K && plan.mode_b == LOAD_VEC_K && l_k_affine
                      && l_sk_a == 1 && l_sk_b == 1 && l_size_k % 16 == 0 && l_size_k >= 96
                      && l_size_k <= 4096 && n_tiles( plan.tile ) < l_cus
                      && ( l_t32 >= l_cus / 2 || l_size_k <= 512 ) && l_t32 <= ( l_size_k < 112 ? 1 : 2 ) * l_cus
                      && std::getenv( "ETIR_NO_KWAVE" ) == nullptr;
    if( l_kw_ok ) {
      // 8 waves up to K = 512, 16 above (config 1, K = 512: 7.58-7.65 us with
      // 8 waves against 7.85-7.87 with 16 and 8.8 with 4; K = 256 and 1024:
      // 8 and 16 equal within 1 %)
      int32_t const l_w = ( l_size_k <= 512 ) ? 8 : 16;
      plan.tile = TILE_F32_KWAVE_32x32;
      plan.tile_fallback = TILE_F32_64x64;
      plan.kwave_waves = l_w;
      plan.kwave_kw = (int32_t) ( ( ( l_size_k + l_w - 1 ) / l_w + 15 ) / 16 * 16 );
      tile_shape( plan.tile, l_bm, l_bn );
    }
  }

  // ------------------------------------------------------------- split K
  // Few output tiles and a long K leave most CUs idle (e.g. an einsum-tree
  // node with M = 64, N = 1024, K = 32768).  Then the outermost K loops (one
  // of them factored if needed) become C loops of a partial contraction that
  // writes one workspace slice per split, and split_reduce sums the slices.
  if( allow_split && !l_f64 && !l_cpx && l_size_k >= 512 && plan.tile != TILE_F32_KWAVE_32x32
      && plan.tile != TILE_GEMV && plan.tile != TILE_SKINNY && plan.tile != TILE_PANEL ) {
    int64_t const l_tiles = n_tiles( plan.tile );
    if( l_tiles > 0 && l_tiles < l_cus ) {
      // at least 128 k per split; aim for two workgroups per CU
      int64_t const l_smax   = l_size_k / 128;
      int64_t const l_target = std::min( ( 2 * l_cus + l_tiles - 1 ) / l_tiles, l_smax );
      std::vector< Loop > l_kk = l_k;          // K loops, outer -> inner
      std::vector< Loop > l_sp;                // split parts, outer -> inner
      int64_t l_sf = 1;
      bool const l_vec_k = plan.mode_a != LOAD_SCALAR && plan.mode_b != LOAD_SCALAR
                        && ( plan.mode_a == LOAD_VEC_K || plan.mode_b == LOAD_VEC_K );
      std::size_t l_i = 0;
      while( l_sf < l_target && l_i < l_kk.size() ) {
        Loop & l_lp = l_kk[l_i];
        int64_t const l_need = ( l_target + l_sf - 1 ) / l_sf;
        // factor of this loop: the smallest divisor that reaches the target,
        // else the largest one that stays within l_smax
        // (first pass: only factors that leave the K of a split a multiple of
        // l_q, so that its rows stay loadable in vectors: 4620 = 4 x 1155 on
        // the fp32 direct-to-LDS kernel measured 457 us, 5 x 924 the vector
        // loads; bf16 2384 = 4 x 596 gathers element by element, 2 x 1192 not;
        // fp32 loops that run on in memory 8-byte vectors at least: 136 x 792
        // x (54 x 18) 11.9 us in 6 x 162, 14.2 in 3 x 324)
        int64_t l_in = 1;                        // K of the loops inside this one
        for( std::size_t l_j = l_i + 1; l_j < l_kk.size(); l_j++ ) l_in *= l_kk[l_j].size;
        int64_t l_q = 1;
        if( l_in == 1 && l_lp.size % 4 == 0 && ( l_lp.s[T_L] == 1 || l_lp.s[T_R] == 1 ) ) l_q = 4;
        if( l_vec_k ) l_q = std::max( l_q, l_f32 ? int64_t( 2 ) : l_vk );
        int64_t l_f = 0;
        for( int l_pass = l_q > 1 ? 0 : 1; l_pass < 2 && l_f == 0; l_pass++ ) {
          for( int64_t l_d = 2; l_d <= l_lp.size; l_d++ ) {
            if( l_lp.size % l_d != 0 || l_sf * l_d > l_smax ) continue;
            if( l_pass == 0 && ( l_lp.size / l_d * l_in ) % l_q != 0 ) continue;
            l_f = l_d;
            if( l_d >= l_need ) break;
          }
          // giving up vector loads pays from 8 splits on (bf16: and a K of
          // 4096), in fp32 also from 4 on where the operands are small (split /
          // whole, bf16 256 x 256: K = 2056 in 2 80 / 16 us, in 8 20 / 16, 4184
          // in 8 34 / 42, 16408 in 14 99 / 146; fp32 in 4, 128 x 128: K = 2092
          // 41 / 50, 4252 77 / 98, 6044 188 / 138; 256 x 256: 2092 44 / 50, 3028
          // 82 / 71; 512 x 384: 2092 63 / 50)
          if( l_pass == 1 && l_vec_k ) {
            int64_t const l_s   = l_sf * l_f;
            int64_t const l_out = l_size_c * l_size_m * l_size_n;
            bool const l_pays = l_f32 ? l_s >= 8 || (    l_s >= 4 && l_out <= 65536
                                                     && l_size_k < ( l_out <= 16384 ? 4608 : 2560 ) )
                                      : l_s >= 8 && l_size_k >= 4096;
            if( !l_pays ) l_f = 0;
          }
        }
        if( l_f == 0 ) break;
        if( l_f == l_lp.size ) {
          l_sp.push_back( l_lp );
          l_sf *= l_lp.size;
          l_lp.size = 1;
          l_i++;
        }
        else {
          // k = ko * (size / f) + ki: the outer part steps over size / f
          Loop l_outer = l_lp;
          int64_t const l_inner = l_lp.size / l_f;
          l_outer.size = l_f;
          for( int l_t = 0; l_t < 4; l_t++ ) l_outer.s[l_t] *= l_inner;
          l_lp.size = l_inner;
          l_sp.push_back( l_outer );
          l_sf *= l_f;
          break;
        }
      }
      // extent of the output (elements) over its C, M and N loops; the
      // workspace slices lie l_span apart, the extent rounded up to 64
      // elements (16-byte aligned slices)
      int64_t l_ext = 1;
      for( auto const * l_set : { &l_c, &l_m, &l_n } ) {
        for( Loop const & l_x : *l_set ) l_ext += ( l_x.size - 1 ) * l_x.s[T_OUT];
      }
      int64_t const l_span = ( l_ext + 63 ) / 64 * 64;
      // dense output: its loops, by output stride, each stride the product
      // of the sizes below it (then the offsets are exactly 0 .. l_ext - 1)
      int64_t l_dense = 0;
      {
        std::vector< std::pair< int64_t, int64_t > > l_ds;
        for( auto const * l_set : { &l_c, &l_m, &l_n } ) {
          for( Loop const & l_x : *l_set ) if( l_x.size > 1 ) l_ds.push_back( { l_x.s[T_OUT], l_x.size } );
        }
        std::sort( l_ds.begin(), l_ds.end() );
        int64_t l_pack = 1;
        bool l_ok = true;
        for( auto const & l_d : l_ds ) {
          l_ok = l_ok && ( l_d.first == l_pack );
          l_pack *= l_d.second;
        }
        if( l_ok && l_pack == l_ext ) l_dense = l_ext;
      }
      // with an aux tensor: every loop either matches the output's stride in
      // the aux tensor or is broadcast (aux stride 0), the broadcast loops
      // outermost in the output; then the aux offset is o % (the extent of
      // the others)
      int64_t l_dense_aux = 0;
      if( l_dense > 0 && plan.needs_aux ) {
        int64_t l_inner = 1;
        int64_t l_bmin = std::numeric_limits< int64_t >::max();
        int64_t l_kmax = 0;
        bool l_ok = true;
        for( auto const * l_set : { &l_c, &l_m, &l_n } ) {
          for( Loop const & l_x : *l_set ) {
            if( l_x.size <= 1 ) continue;
            if( l_x.s[T_AUX] == 0 ) l_bmin = std::min( l_bmin, l_x.s[T_OUT] );
            else {
              l_ok = l_ok && ( l_x.s[T_AUX] == l_x.s[T_OUT] );
              l_inner *= l_x.size;
              l_kmax = std::max( l_kmax, l_x.s[T_OUT] );
            }
          }
        }
        if( l_ok && ( l_bmin == std::numeric_limits< int64_t >::max() || l_bmin == l_inner ) && l_kmax < l_inner ) {
          l_dense_aux = l_inner;
        }
      }
      int64_t const l_ws_bytes = 4 * l_sf * l_span;
      if( l_sf >= 2 && l_size_k / l_sf >= 128 && l_ws_bytes <= ( int64_t( 1 ) << 29 ) ) {
        // loop arrays of the partial contraction
        std::vector< int32_t > l_pt;
        std::vector< int64_t > l_psz, l_pl, l_pr, l_pa, l_po;
        auto add = [&]( int32_t t, int64_t sz, int64_t sl, int64_t sr, int64_t sa, int64_t so ) {
          l_pt.push_back( t ); l_psz.push_back( sz ); l_pl.push_back( sl ); l_pr.push_back( sr );
          l_pa.push_back( sa ); l_po.push_back( so );
        };
        int64_t l_inner_sp = 1;
        for( std::size_t l_j = l_sp.size(); l_j-- > 0; ) {
          Loop const & l_x = l_sp[l_j];
          add( ETIR_DIM_C, l_x.size, l_x.s[T_L], l_x.s[T_R], 0, l_span * l_inner_sp );
          l_inner_sp *= l_x.size;
        }
        for( auto const * l_set : { &l_c, &l_m, &l_n } ) {
          for( Loop const & l_x : *l_set ) add( l_x.type, l_x.size, l_x.s[T_L], l_x.s[T_R], l_x.s[T_AUX], l_x.s[T_OUT] );
        }
        for( Loop const & l_x : l_kk ) {
          if( l_x.size > 1 ) add( ETIR_DIM_K, l_x.size, l_x.s[T_L], l_x.s[T_R], 0, 0 );
        }
        auto l_part = std::make_shared< ContractionPlan >();
        int l_err = plan_contraction_impl( (int64_t) l_pt.size(), l_pt.data(), l_psz.data(), l_pl.data(),
                                           l_pr.data(), l_pa.data(), l_po.data(), dtype_left, dtype_right,
                                           ETIR_FP32, ETIR_FP32, ETIR_KTYPE_ZERO, ETIR_KTYPE_MADD,
                                           ETIR_KTYPE_UNDEFINED, false, *l_part, place, dry, copied );
        if( l_err != ETIR_SUCCESS ) {
          release_contraction( *l_part );
          return l_err;
        }
        plan.args.k_affine = l_part->args.k_affine;
        if( dry ) {
          plan.split  = (int32_t) l_sf;
          plan.C      = l_size_c;
          plan.M      = l_part->M;
          plan.N      = l_part->N;
          plan.K      = l_size_k;
          plan.mode_a = l_part->mode_a;
          plan.mode_b = l_part->mode_b;
          plan.tile   = l_part->tile;
          return ETIR_SUCCESS;
        }
        if( place != nullptr ) {
          l_err = place_take( *place, (std::size_t) l_ws_bytes, &plan.d_ws, "split-K workspace" );
          if( l_err != ETIR_SUCCESS ) {
            release_contraction( *l_part );
            return l_err;
          }
        }
        else {
          hipError_t l_he = hipMalloc( &plan.d_ws, (std::size_t) l_ws_bytes );
          if( l_he != hipSuccess ) {
            plan.d_ws = nullptr;
            release_contraction( *l_part );
            return fail( ETIR_UNDEFINED_ERROR, std::string( "contraction: workspace allocation failed: " )
                                               + hipGetErrorString( l_he ) );
          }
        }
        plan.split    = (int32_t) l_sf;
        plan.out_span = l_span;
        plan.out_dense     = ( !plan.needs_aux || l_dense_aux > 0 ) ? l_dense : 0;
        plan.out_dense_aux = plan.needs_aux ? l_dense_aux : 0;
        plan.partial  = l_part;
        plan.C = l_size_c;
        plan.M = l_part->M;
        plan.N = l_part->N;
        plan.K = l_size_k;
        plan.mode_a = l_part->mode_a;
        plan.mode_b = l_part->mode_b;
        plan.tile = l_part->tile;
        plan.flops = 2 * l_size_c * l_size_m * l_size_n * l_size_k;
        int64_t const l_esz_o = ( dtype_out == ETIR_BF16 ) ? 2 : 4;
        plan.bytes = l_esz * l_size_c * ( l_size_m + l_size_n ) * l_size_k
                   + l_esz_o * l_size_c * l_size_m * l_size_n;
        plan.desc = "split-K S=" + std::to_string( l_sf ) + " K'=" + std::to_string( l_size_k / l_sf )
                  + " | " + l_part->desc + " | reduce" + ( plan.out_dense > 0 ? " flat" : "" );
        return ETIR_SUCCESS;
      }
    }
  }
  if( l_big_k_split && plan.tile == TILE_F32_DMA_128x128 ) {
    // K did not split (and K over waves did not take the node): back to the
    // tile that fills the chip by itself
    plan.tile = l_tile_unsplit;
    tile_shape( plan.tile, l_bm, l_bn );
  }

  plan.C = l_size_c;
  plan.M = l_kern_m;
  plan.N = l_kern_n;
  plan.K = l_size_k;
  plan.args.k_affine = l_k_affine ? 1 : 0;
  if( dry ) return ETIR_SUCCESS;
  // complex: four real products per complex multiply-add
  plan.flops = ( l_cpx ? 8 : 2 ) * l_size_c * l_size_m * l_size_n * l_size_k;
  int64_t const l_esz_out = ( dtype_out == ETIR_BF16 ) ? 2 : ( dtype_out == ETIR_FP64 ? 8 : 4 );
  bool const l_read_out = ktype_first_touch == ETIR_KTYPE_ADD || ktype_first_touch == ETIR_KTYPE_UNDEFINED;
  plan.bytes = ( l_cpx ? 2 : 1 )
             * (   l_esz * l_size_c * ( l_size_m + l_size_n ) * l_size_k
                 + l_esz_out * l_size_c * l_size_m * l_size_n * ( 1 + ( l_read_out ? 1 : 0 )
                                                                    + ( plan.needs_aux ? 1 : 0 ) ) );

  std::ostringstream l_d;
  l_d << "contract " << tile_str( plan.tile )
      << " C=" << l_size_c << dims_str( l_c )
      << " M=" << plan.M << dims_str( l_km )
      << " N=" << plan.N << dims_str( l_kn )
      << " K=" << plan.K << dims_str( l_k )
      << " A=" << ( l_swap ? "right" : "left" ) << ":" << mode_str( plan.mode_a )
      << " B=" << ( l_swap ? "left" : "right" ) << ":" << mode_str( plan.mode_b )
      << " k_affine=" << ( l_k_affine ? 1 : 0 );
  plan.desc = l_d.str();

  // ------------------------------------------------------ device tables
  // layout: int64 C tables first (8-byte aligned), then int32 tables
  std::vector< int64_t > l_c64;
  l_c64.insert( l_c64.end(), l_tc_a.begin(),   l_tc_a.end() );
  l_c64.insert( l_c64.end(), l_tc_b.begin(),   l_tc_b.end() );
  l_c64.insert( l_c64.end(), l_tc_aux.begin(), l_tc_aux.end() );
  l_c64.insert( l_c64.end(), l_tc_out.begin(), l_tc_out.end() );
  std::vector< int32_t > l_t32;
  auto app32 = [&]( std::vector< int64_t > const & t ) {
    for( int64_t l_v : t ) l_t32.push_back( (int32_t) l_v );
  };
  std::size_t const l_o_tm_a = l_t32.size(); app32( l_tm_a );
  std::size_t const l_o_tm_x = l_t32.size(); app32( l_tm_aux );
  std::size_t const l_o_tm_o = l_t32.size(); app32( l_tm_out );
  std::size_t const l_o_tn_b = l_t32.size(); app32( l_tn_b );
  std::size_t const l_o_tn_x = l_t32.size(); app32( l_tn_aux );
  std::size_t const l_o_tn_o = l_t32.size(); app32( l_tn_out );
  std::size_t const l_o_tk_a = l_t32.size(); app32( l_tk_a );
  std::size_t const l_o_tk_b = l_t32.size(); app32( l_tk_b );

  std::size_t const l_bytes64 = l_c64.size() * sizeof( int64_t );
  std::size_t const l_bytes32 = l_t32.size() * sizeof( int32_t );
  std::size_t const l_total = l_bytes64 + l_bytes32 + 256;
  char * l_base = nullptr;
  if( place != nullptr ) {
    // caller's region: the tables are generated there by a kernel from the
    // same loops (and slots) the host enumerated them from above
    int l_err = place_take( *place, l_total, &plan.d_tables, "offset tables" );
    if( l_err != ETIR_SUCCESS ) return l_err;
    l_base = reinterpret_cast< char * >( plan.d_tables );
    int64_t const l_b = int64_t( l_base - place->base );
    int64_t const l_o32 = l_b + int64_t( l_bytes64 );
    auto fill = [&]( std::vector< Loop > const & dims, std::initializer_list< int > slots,
                     std::initializer_list< int64_t > dst, bool is64 ) -> int {
      if( (int) dims.size() > kFillMaxDims ) {
        return fail( ETIR_COMPILATION_FAILED, "contraction: too many fused loops of one type for the "
                                              "allocation-free entry point" );
      }
      TableFill l_f{};
      l_f.count = 1;
      for( Loop const & l_x : dims ) l_f.count *= l_x.size;
      l_f.ndims = (int32_t) dims.size();
      l_f.ntab = (int32_t) slots.size();
      l_f.is64 = is64 ? 1 : 0;
      for( int l_d = 0; l_d < l_f.ndims; l_d++ ) l_f.sizes[l_d] = dims[l_d].size;
      int l_t = 0;
      for( int l_sl : slots ) {
        for( int l_d = 0; l_d < l_f.ndims; l_d++ ) l_f.strides[l_t][l_d] = dims[l_d].s[l_sl];
        l_t++;
      }
      l_t = 0;
      for( int64_t l_o : dst ) l_f.dst[l_t++] = l_o;
      if( l_f.count == 0 ) return ETIR_SUCCESS;
      return launch_fill_tables( l_f, place->base, place->stream );
    };
    int64_t const l_cs = int64_t( sizeof( int64_t ) ) * l_size_c;
    int l_err2 = fill( l_c, { l_sa, l_sb, T_AUX, T_OUT }, { l_b, l_b + l_cs, l_b + 2 * l_cs, l_b + 3 * l_cs }, true );
    if( l_err2 == ETIR_SUCCESS ) {
      l_err2 = fill( l_km, { l_sa, T_AUX, T_OUT }, { l_o32 + 4 * int64_t( l_o_tm_a ), l_o32 + 4 * int64_t( l_o_tm_x ),
                                                    l_o32 + 4 * int64_t( l_o_tm_o ) }, false );
    }
    if( l_err2 == ETIR_SUCCESS ) {
      l_err2 = fill( l_kn, { l_sb, T_AUX, T_OUT }, { l_o32 + 4 * int64_t( l_o_tn_b ), l_o32 + 4 * int64_t( l_o_tn_x ),
                                                    l_o32 + 4 * int64_t( l_o_tn_o ) }, false );
    }
    if( l_err2 == ETIR_SUCCESS ) {
      l_err2 = fill( l_k, { l_sa, l_sb }, { l_o32 + 4 * int64_t( l_o_tk_a ), l_o32 + 4 * int64_t( l_o_tk_b ) }, false );
    }
    if( l_err2 != ETIR_SUCCESS ) return l_err2;
  }
  else {
    ETIR_HIP_CHECK( hipMalloc( &plan.d_tables, l_total ) );
    l_base = reinterpret_cast< char * >( plan.d_tables );
    hipError_t l_e1 = hipMemcpy( l_base, l_c64.data(), l_bytes64, hipMemcpyHostToDevice );
    hipError_t l_e2 = l_bytes32 > 0
                    ? hipMemcpy( l_base + l_bytes64, l_t32.data(), l_bytes32, hipMemcpyHostToDevice )
                    : hipSuccess;
    if( l_e1 != hipSuccess || l_e2 != hipSuccess ) {
      (void) hipFree( plan.d_tables );
      plan.d_tables = nullptr;
      return fail( ETIR_UNDEFINED_ERROR, "contraction: copying offset tables to the device failed" );
    }
  }

  ContractArgs & a = plan.args;
  a = ContractArgs();
  int64_t const * l_p64 = reinterpret_cast< int64_t const * >( l_base );
  a.tc_a   = l_p64;
  a.tc_b   = l_p64 + l_size_c;
  a.tc_aux = l_p64 + 2 * l_size_c;
  a.tc_out = l_p64 + 3 * l_size_c;
  int32_t const * l_p32 = reinterpret_cast< int32_t const * >( l_base + l_bytes64 );
  a.tm_a   = l_p32 + l_o_tm_a;
  a.tm_aux = l_p32 + l_o_tm_x;
  a.tm_out = l_p32 + l_o_tm_o;
  a.tn_b   = l_p32 + l_o_tn_b;
  a.tn_aux = l_p32 + l_o_tn_x;
  a.tn_out = l_p32 + l_o_tn_o;
  a.tk_a   = l_p32 + l_o_tk_a;
  a.tk_b   = l_p32 + l_o_tk_b;
  a.M = (int32_t) l_kern_m;
  a.N = (int32_t) l_kern_n;
  a.K = (int32_t) l_size_k;
  a.C = (int32_t) l_size_c;
  {
    // a C dim innermost in the output: each workgroup (one C index) would
    // write every C-th element, and the workgroups holding the other C
    // indices of the same output lines would run far apart in time; with C
    // fastest in the workgroup order they run side by side (same XCD, same
    // L2) and complete those lines there
    int64_t l_min_c = std::numeric_limits< int64_t >::max();
    int64_t l_min_mn = std::numeric_limits< int64_t >::max();
    for( Loop const & l_x : l_c ) if( l_x.size > 1 ) l_min_c = std::min( l_min_c, l_x.s[T_OUT] );
    for( auto const * l_set : { &l_m, &l_n } ) {
      for( Loop const & l_x : *l_set ) if( l_x.size > 1 ) l_min_mn = std::min( l_min_mn, l_x.s[T_OUT] );
    }
    a.c_inner = ( l_size_c > 1 && l_min_c < l_min_mn ) ? 1 : 0;
    if( a.c_inner ) plan.desc += " c_inner";
  }
  a.tiles_m = (int32_t) ( ( l_kern_m + l_bm - 1 ) / l_bm );
  a.tiles_n = (int32_t) ( ( l_kern_n + l_bn - 1 ) / l_bn );
  a.k_affine = l_k_affine ? 1 : 0;
  a.sk_a = (int32_t) l_sk_a;
  a.sk_b = (int32_t) l_sk_b;
  a.first_touch = ktype_first_touch;
  a.last_touch  = ktype_last_touch;
  a.out_bf16 = ( dtype_out == ETIR_BF16 ) ? 1 : 0;
  a.out_v8 = ( dtype_out == ETIR_BF16 && runs_contiguous( l_tn_out, 8, 8 ) && all_multiple( l_tm_out, 8 )
               && all_multiple( l_tc_out, 8 ) ) ? 1 : 0;
  // start-time stagger of the persistent direct-to-LDS kernel: 4 phases, 3
  // units (~3 us) apart (measured on config 3; diagnostic override by env)
  a.dma_phases = 4;
  a.dma_stagger = 3;
  if( char const * l_env = std::getenv( "ETIR_DMA_PHASES" ) ) a.dma_phases = std::atoi( l_env );
  if( char const * l_env = std::getenv( "ETIR_DMA_STAGGER" ) ) a.dma_stagger = std::atoi( l_env );
  auto affine_stride = []( std::vector< int64_t > const & t ) -> int32_t {
    int64_t const l_st = t.size() > 1 ? t[1] : 0;
    for( std::size_t l_i = 0; l_i < t.size(); l_i++ ) {
      if( t[l_i] != int64_t( l_i ) * l_st ) return -1;
    }
    return ( l_st >= 0 && l_st <= std::numeric_limits< int32_t >::max() ) ? int32_t( l_st ) : -1;
  };
  a.sm_a   = affine_stride( l_tm_a );
  a.sn_b   = affine_stride( l_tn_b );
  a.sm_out = affine_stride( l_tm_out );
  a.sn_out = affine_stride( l_tn_out );
  a.gemv_v4 = ( plan.tile == TILE_GEMV && l_tm_out.size() == 1 && l_tn_out.size() % 4 == 0 && a.sn_b == 1
                && a.sn_out == 1 && all_multiple( l_tc_b, 4 ) && all_multiple( l_tk_b, 4 )
                && all_multiple( l_tc_out, 4 ) && all_multiple( l_tm_out, 4 ) ) ? 1 : 0;
  if( a.gemv_v4 ) plan.desc += " v4";
  {
    bool const l_short_a = l_kern_m <= l_kern_n;
    std::vector< int64_t > const & l_tl = l_short_a ? l_tn_b : l_tm_a;
    std::vector< int64_t > const & l_tcl = l_short_a ? l_tc_b : l_tc_a;
    int64_t const l_skl = l_short_a ? l_sk_b : l_sk_a;
    a.skinny_kvec = ( plan.tile == TILE_SKINNY && l_k_affine && ( l_size_k <= 1 || l_skl == 1 ) && l_size_k % 4 == 0
                      && all_multiple( l_tl, 4 ) && all_multiple( l_tcl, 4 ) ) ? 1 : 0;
    if( a.skinny_kvec ) plan.desc += " kvec";
    // the output as [long][short] with the short side unit-stride (short
    // offsets s, long offsets i * S): a workgroup's outputs are one block,
    // written in address order through LDS; only where the output is
    // written, not read (no accumulation, no aux)
    std::vector< int64_t > const & l_tlo = l_short_a ? l_tn_out : l_tm_out;
    std::vector< int64_t > const & l_tso = l_short_a ? l_tm_out : l_tn_out;
    a.skinny_blk = 0;
    if( plan.tile == TILE_SKINNY && ktype_first_touch == ETIR_KTYPE_ZERO && !plan.needs_aux
        && ( ktype_last_touch == ETIR_KTYPE_UNDEFINED || ktype_last_touch == ETIR_KTYPE_RELU )
        && affine_stride( l_tso ) == 1 ) {
      int64_t const l_s = int64_t( l_tso.size() );
      bool l_ok = true;
      for( std::size_t l_i = 0; l_ok && l_i < l_tlo.size(); l_i++ ) l_ok = ( l_tlo[l_i] == int64_t( l_i ) * l_s );
      if( l_ok ) {
        a.skinny_blk = 1;
        plan.desc += " blk";
      }
    }
  }
  if( l_cpx ) {
    a.cpx_a   = l_x[0].s[l_sa];
    a.cpx_b   = l_x[0].s[l_sb];
    a.cpx_out = l_x[0].s[T_OUT];
  }
  {
    int64_t l_mo = 0, l_no = 0;
    for( int64_t l_v : l_tm_out ) l_mo = std::max( l_mo, l_v );
    for( int64_t l_v : l_tn_out ) l_no = std::max( l_no, l_v );
    a.out_off32 = ( 4 * ( l_mo + l_no ) + 4 < ( int64_t( 1 ) << 32 ) ) ? 1 : 0;
    // non-temporal output stores only where each store instruction of the
    // fast epilogue (32 consecutive columns per half-wave) writes whole
    // unit-stride runs: the output's columns are consecutive in groups of 32
    a.out_nt = ( l_run_n >= 32 && ( l_run_n % 32 == 0 || l_run_n == l_tn_out.size() ) ) ? 1 : 0;
    if( char const * l_env = std::getenv( "ETIR_OUT_NT" ) ) a.out_nt = std::atoi( l_env ) != 0 ? 1 : 0;
  }
  // K of one step with plain output: the one-step form of the fp32
  // direct-to-LDS kernel; there, short output runs whose rows are neighbours
  // in the output leave by whole runs.  Otherwise for rows of whole 128-byte
  // lines (20000 x 512 x 32: 14.9 -> 13.4 us; rows of 4100 columns, whose
  // streamed lines are cut in two, 27.1 -> 28.4 us)
  bool const l_one_step = plan.tile == TILE_F32_DMA_128x128 && l_k_affine && l_size_k <= 32 && a.out_off32
                       && ktype_first_touch == ETIR_KTYPE_ZERO
                       && ( ktype_last_touch == ETIR_KTYPE_UNDEFINED || ktype_last_touch == ETIR_KTYPE_RELU );
  bool const l_by_runs = l_one_step && l_run_n >= 8 && l_run_n < 32 && l_run_n % 4 == 0
                      && runs_contiguous( l_tn_out, (int64_t) l_run_n, 4 ) && all_multiple( l_tm_out, 4 )
                      && all_multiple( l_tc_out, 4 ) && l_tm_out.size() > 1
                      && l_tm_out[1] == l_tm_out[0] + (int64_t) l_run_n;
  a.k_one_step = ( l_by_runs || ( l_one_step && all_multiple( l_tm_out, 32 ) && all_multiple( l_tc_out, 32 ) ) ) ? 1 : 0;
  if( a.k_one_step ) plan.desc += " one_step";
  a.out_run = 0;
  a.n_step = 0;
  if( l_by_runs ) {
    a.out_run = int32_t( l_run_n );
    a.n_step  = int32_t( 128 / l_run_n * l_run_n );
    a.tiles_n = (int32_t) ( ( l_kern_n + a.n_step - 1 ) / a.n_step );
    plan.desc += " runs=" + std::to_string( l_run_n );
  }
  if( plan.tile == TILE_PANEL ) {
    int64_t l_mo = 0, l_no = 0;
    for( int64_t l_v : l_tm_out ) l_mo = std::max( l_mo, l_v );
    for( int64_t l_v : l_tn_out ) l_no = std::max( l_no, l_v );
    a.out_bytes  = uint32_t( 4 * ( l_mo + l_no + 1 ) );
    a.panel_grid = int32_t( l_cus );
  }
  if( plan.tile == TILE_BF16_DMA_256x256 && plan.dma_variant == 3 && persistent_dma_eligible( a, 256, 256 ) ) {
    plan.desc += " persistent";
  }
  return ETIR_SUCCESS;
}

// Rate (TFLOP/s) a plan's kernel reaches on a full chip, by its tile and its
// operands' load modes (one or both gathered element by element), measured at
// 511 to 4095 a side.  `far`: a gathered operand above an XCD's 4 MB L2 whose
// neighbouring elements are neither along K nor along its rows (measured at
// 1152 to 8064 a side).  Only for comparing a plan with its packed forms.
double plan_rate( ContractionPlan const & plan, bool far ) {
  int const l_s = ( plan.mode_a == LOAD_SCALAR ? 1 : 0 ) + ( plan.mode_b == LOAD_SCALAR ? 1 : 0 );
  auto by_mode = [&]( double vec, double one, double two, double far_one ) {
    return l_s == 0 ? vec : ( far ? far_one : ( l_s == 1 ? one : two ) );
  };
  switch( plan.tile ) {
    case TILE_F32_DMA_128x128:  return 135.0;
    case TILE_F32_128x128:      return by_mode( 112.0, 75.0, 75.0, 16.0 );
    case TILE_F32_64x64:        return by_mode( 78.0, plan.args.k_affine && plan.split > 1 ? 36.0 : 30.0, 25.0, 25.0 );
    case TILE_F32_KWAVE_32x32:  return 50.0;
    case TILE_BF16_DMA_256x256: return 1100.0;
    case TILE_BF16_DMA_128x128: return 850.0;
    case TILE_BF16_256x128:     return by_mode( 550.0, 100.0, 95.0, 20.0 );
    case TILE_BF16_128x128:     return by_mode( 550.0, plan.args.k_affine ? 80.0 : 50.0, 45.0, 20.0 );
    case TILE_BF16_64x64:       return by_mode( 300.0, 46.0, 45.0, 25.0 );
    case TILE_F64_64x64:        return by_mode( plan.args.k_affine ? 48.0 : 41.0, 46.0, 46.0, 18.0 );
    case TILE_F64_DMA_128x128:  return 68.0;
    default:                    return 0.0;   // not a tile that packing is weighed against
  }
}

// estimated time (us): flops at plan_rate over the useful part of the tile
// grid, or the tensors' bytes at 3.5 TB/s (a scattered output at 2) where that
// is longer.  fp64 tiles run in whole rounds of one per CU (2100 a side, 289
// tiles of 128 x 128, takes as long as 2500 with 400)
double plan_us( ContractionPlan const & plan, bool far, double flops, double bytes_in, double bytes_out ) {
  int64_t l_bm, l_bn;
  tile_shape( plan.tile, l_bm, l_bn );
  double const l_tm = double( ( plan.M + l_bm - 1 ) / l_bm ), l_tn = double( ( plan.N + l_bn - 1 ) / l_bn );
  double const l_tiles = l_tm * l_tn * double( plan.C ) * double( plan.split );
  bool const l_f64 = plan.tile == TILE_F64_64x64 || plan.tile == TILE_F64_DMA_128x128;
  double const l_util = double( plan.M ) * double( plan.N ) / ( l_tm * double( l_bm ) * l_tn * double( l_bn ) )
                      * ( l_f64 ? l_tiles / ( 256.0 * std::ceil( l_tiles / 256.0 ) ) : std::min( 1.0, l_tiles / 256.0 ) );
  return std::max( flops / ( plan_rate( plan, far ) * l_util * 1e6 ),
                   bytes_in / 3.5e6 + bytes_out / ( plan.scattered ? 2.0e6 : 3.5e6 ) ) + 5.0;
}

// Weighs copying one or both operands K-contiguous into a workspace
// (O((M + N) K) bytes) against reading them in place (O(M N K) loads), and
// builds the packed contraction where it is clearly faster.
//
// In place, an operand without 16-byte runs along its rows or along the K
// order of the other one is gathered element by element; a K-contiguous copy
// (rows padded with zeros to whole 16-byte vectors when both are copied) takes
// the vector tiles and the direct-to-LDS kernels.  A K of several loops that
// are not adjacent in an operand (table K: 112 against 135 TFLOP/s in fp32)
// is packed too where the longer kernel pays for the copy.  Measured, in
// place against packed, copies included:
//   aecf,bfde->abcd 96,96,84,84,84,84 fp32 (left contiguous along f, right
//     along e)                               62.3 -> 7.38 ms (14.7 -> 124 TFLOP/s)
//   the same, 48,48,42,42,42,42 fp64          795 -> 324 us
//   acd,dbc->ab 384,376,376,384 fp32         1949 -> 466 us
//   mk,nk->mn, 767 / 1023 / 2047 a side       fp32 61 -> 31, 80 -> 44, 371 -> 160 us
//                                             bf16 44 -> 23, 58 -> 25, 370 -> 59 us
// and packed where the rule keeps them in place (a copy costs about 7 us
// beside its bytes): aecf,bfde->abcd 24,24,12,12,12,12 fp32 12.5 -> 14.0 us,
// eafd,fbec->abcd 42,42,21,21,21,21 fp32 46 -> 53 us.
//
// Never fails: without a gain, or where the copies would take more than an
// eighth of the free device memory, the plan stays as it is.
void try_pack( int64_t            num_loops,
               int32_t const    * dim_types,
               int64_t const    * sizes,
               int64_t const    * strides_left,
               int64_t const    * strides_right,
               int64_t const    * strides_out_aux,
               int64_t const    * strides_out,
               int32_t            dtype_left,
               int32_t            dtype_right,
               int32_t            dtype_comp,
               int32_t            dtype_out,
               int32_t            ktype_first_touch,
               int32_t            ktype_main,
               int32_t            ktype_last_touch,
               bool               allow_split,
               ContractionPlan  & plan ) {
  if( ktype_main != ETIR_KTYPE_MADD || std::getenv( "ETIR_TILE" ) != nullptr ) return;
  // a side of up to 32 reads the other operand once or twice: a copy of it
  // reads it as often (efbadx,cfx->abcdex, N = 24: 23.2 ms in place, 25.0 packed)
  if( std::min( plan.M, plan.N ) <= 32 ) return;
  if( plan.C <= 0 || plan.M <= 0 || plan.N <= 0 || plan.K <= 1 || plan_rate( plan, false ) == 0.0 ) return;
  auto in_vec = [&]( int32_t m ) { return m == LOAD_VEC_MN || m == LOAD_VEC_K; };
  bool const l_affine = plan.args.k_affine != 0;
  if( in_vec( plan.mode_a ) && in_vec( plan.mode_b ) && l_affine && !plan.scattered
      && plan.tile != TILE_F64_64x64 ) {
    return;
  }

  int64_t const   l_esz  = dtype_bytes( dtype_left );
  int64_t const   l_vk   = 16 / l_esz;
  int64_t const * l_st[2] = { strides_left, strides_right };

  // loops an operand runs over (size-1 loops and broadcast ones do not move it)
  struct Dim { int64_t size, s, id; };
  std::vector< Dim > l_rows[2], l_k[2];     // C and row loops; K loops: by the operand's stride, outer first
  double l_bytes[2];
  for( int l_op = 0; l_op < 2; l_op++ ) {
    int64_t l_n = 1;
    for( int64_t l_lo = 0; l_lo < num_loops; l_lo++ ) {
      if( sizes[l_lo] <= 1 || dim_types[l_lo] == ETIR_DIM_I || dim_types[l_lo] == ETIR_DIM_J ) continue;
      if( dim_types[l_lo] == ( l_op == 0 ? ETIR_DIM_N : ETIR_DIM_M ) ) continue;
      bool const l_is_k = dim_types[l_lo] == ETIR_DIM_K;
      if( l_st[l_op][l_lo] == 0 ) {
        if( l_is_k ) return;                // a K loop that an operand does not move along
        continue;
      }
      ( l_is_k ? l_k : l_rows )[l_op].push_back( { sizes[l_lo], l_st[l_op][l_lo], l_lo } );
      l_n *= sizes[l_lo];
    }
    for( auto * l_set : { &l_rows[l_op], &l_k[l_op] } ) {
      std::stable_sort( l_set->begin(), l_set->end(), []( Dim const & x, Dim const & y ) { return x.s > y.s; } );
    }
    l_bytes[l_op] = double( l_n ) * double( l_esz );
  }

  double const l_flops = 2.0 * double( plan.C ) * double( plan.M ) * double( plan.N ) * double( plan.K );
  double const l_out   = double( dtype_bytes( dtype_out ) ) * double( plan.C ) * double( plan.M ) * double( plan.N );
  // a gathered operand whose unit-stride loop is neither the innermost K loop
  // of the plan's K order nor the innermost row loop
  bool l_far = false;
  for( int l_op = 0; l_op < 2; l_op++ ) {
    bool const l_is_a = ( l_op == 0 ) != plan.swapped;
    if( ( l_is_a ? plan.mode_a : plan.mode_b ) != LOAD_SCALAR ) continue;
    // the K order is that of the kernel's A operand when a K loop is its
    // unit-stride one, else that of B when one is B's
    auto unit_k = [&]( int op ) { return !l_k[op].empty() && l_k[op].back().s == 1; };
    int const l_opa = plan.swapped ? 1 : 0;
    int const l_order = unit_k( l_opa ) ? l_opa : ( unit_k( 1 - l_opa ) ? 1 - l_opa : l_opa );
    int64_t const l_kin = l_k[l_order].empty() ? -1 : l_k[l_order].back().id;
    bool l_near = l_kin >= 0 && l_st[l_op][l_kin] == 1;
    for( Dim const & l_d : l_rows[l_op] ) l_near = l_near || ( l_d.s == 1 && dim_types[l_d.id] != ETIR_DIM_C );
    l_far = l_far || ( !l_near && l_bytes[l_op] > 4.0e6 );
  }
  double const l_plain_us = plan_us( plan, l_far, l_flops, l_bytes[0] + l_bytes[1], l_out );
  double const l_limit_us = 0.93 * l_plain_us - 8.0;
  // not worth planning the alternatives: the fastest kernel and one copy
  double const l_top = dtype_left == ETIR_BF16 ? 1100.0 : ( dtype_left == ETIR_FP64 ? 68.0 : 135.0 );
  double const l_small = std::min( l_bytes[0], l_bytes[1] );
  if(    std::max( l_flops / ( l_top * 1e6 ), ( l_bytes[0] + l_bytes[1] + l_out ) / 3.5e6 ) + 13.0
       + 2.0 * l_small / 2.5e6 >= l_limit_us ) {
    return;
  }

  // the alternatives: copy the left, the right, or both
  struct Loops {
    std::vector< int32_t > type;
    std::vector< int64_t > size, s[2], aux, out;
  };
  struct Choice { double us; bool use[2]; Loops loops; int order; int64_t pitch; };
  Choice l_best{ l_limit_us, { false, false }, {}, 0, 0 };
  // row length of the copies where both are made: whole vectors, and where few
  // tiles and a long K ask for a split, the next length that divides into
  // enough parts of whole vectors (bf16 ea,ebcd->abcd 256,4562,99: 4568 = 8 x
  // 571 in 2 parts that gather element by element 179 us)
  int64_t l_pitch = ( plan.K + l_vk - 1 ) / l_vk * l_vk;
  if( allow_split && dtype_left != ETIR_FP64 && plan.K >= 512 ) {
    int64_t const l_t = ( plan.M + 63 ) / 64 * ( ( plan.N + 63 ) / 64 ) * plan.C;
    int64_t const l_parts = l_t < 256 ? std::min( ( 512 + l_t - 1 ) / l_t, plan.K / 128 ) : 1;
    auto divides = [&]( int64_t k ) {
      for( int64_t l_d = l_parts; l_d < 2 * l_parts && l_d * 128 <= k; l_d++ ) {
        if( k % ( l_d * l_vk ) == 0 ) return true;
      }
      return false;
    };
    // (a multiple of l_parts vectors is at most that many vectors away)
    while( !divides( l_pitch ) ) l_pitch += l_vk;
  }
  for( int l_ch = 1; l_ch < 4; l_ch++ ) {
    bool const l_use[2] = { ( l_ch & 1 ) != 0, ( l_ch & 2 ) != 0 };
    bool const l_both = l_use[0] && l_use[1];
    Choice l_c{ 0.0, { l_use[0], l_use[1] }, {}, 0, 0 };
    // K order: that of the operand read in place, or of the larger one
    l_c.order = l_both ? ( l_bytes[0] >= l_bytes[1] ? 0 : 1 ) : ( l_use[0] ? 1 : 0 );
    l_c.pitch = l_both ? l_pitch : plan.K;
    Loops & l_lp = l_c.loops;
    double l_pack_bytes = 0.0;
    std::vector< int64_t > l_packed[2];      // stride per loop of a copied operand
    for( int l_op = 0; l_op < 2; l_op++ ) {
      l_packed[l_op].assign( (std::size_t) num_loops, 0 );
      int64_t l_s = 1;
      for( std::size_t l_i = l_k[l_c.order].size(); l_i-- > 0; ) {
        l_packed[l_op][ l_k[l_c.order][l_i].id ] = l_s;
        l_s *= l_k[l_c.order][l_i].size;
      }
      l_s = l_c.pitch;
      for( std::size_t l_i = l_rows[l_op].size(); l_i-- > 0; ) {
        l_packed[l_op][ l_rows[l_op][l_i].id ] = l_s;
        l_s *= l_rows[l_op][l_i].size;
      }
      if( l_use[l_op] ) l_pack_bytes += double( l_s ) * double( l_esz );
    }
    for( int64_t l_lo = 0; l_lo < num_loops; l_lo++ ) {
      if( sizes[l_lo] <= 1 || dim_types[l_lo] == ETIR_DIM_I || dim_types[l_lo] == ETIR_DIM_J ) continue;
      if( l_both && dim_types[l_lo] == ETIR_DIM_K ) continue;
      l_lp.type.push_back( dim_types[l_lo] );
      l_lp.size.push_back( sizes[l_lo] );
      for( int l_op = 0; l_op < 2; l_op++ ) {
        l_lp.s[l_op].push_back( l_use[l_op] ? l_packed[l_op][l_lo] : l_st[l_op][l_lo] );
      }
      l_lp.aux.push_back( strides_out_aux != nullptr ? strides_out_aux[l_lo] : strides_out[l_lo] );
      l_lp.out.push_back( strides_out[l_lo] );
    }
    if( l_both ) {
      // one K loop over whole vectors: the copies' padding holds zeros
      l_lp.type.push_back( ETIR_DIM_K );
      l_lp.size.push_back( l_c.pitch );
      for( int l_op = 0; l_op < 2; l_op++ ) l_lp.s[l_op].push_back( 1 );
      l_lp.aux.push_back( 0 );
      l_lp.out.push_back( 0 );
    }
    ContractionPlan l_try;
    if( plan_contraction_impl( (int64_t) l_lp.type.size(), l_lp.type.data(), l_lp.size.data(), l_lp.s[0].data(),
                               l_lp.s[1].data(), l_lp.aux.data(), l_lp.out.data(), dtype_left, dtype_right,
                               dtype_comp, dtype_out, ktype_first_touch, ktype_main, ktype_last_touch, allow_split,
                               l_try, nullptr, true, true ) != ETIR_SUCCESS ) {
      continue;
    }
    if( plan_rate( l_try, false ) == 0.0 || !in_vec( l_try.mode_a ) || !in_vec( l_try.mode_b ) ) continue;
    // the copies: 8 us each (launch, and the gap before the kernel that reads
    // it) and 2.5 TB/s, read and written
    l_c.us = plan_us( l_try, false, l_flops, l_bytes[0] + l_bytes[1], l_out ) + 8.0 * ( l_both ? 2.0 : 1.0 )
           + 2.0 * l_pack_bytes / 2.5e6;
    // at most 2 GiB of workspace
    if( l_pack_bytes > double( int64_t( 1 ) << 31 ) ) continue;
    if( l_c.us < l_best.us ) l_best = l_c;
  }
  if( !l_best.use[0] && !l_best.use[1] ) return;

  auto l_pk = std::make_shared< PackedContraction >();
  auto drop = [&]() {
    release_contraction( l_pk->cont );
    for( PermutePlan & l_p : l_pk->perm ) release_permute( l_p );
    if( l_pk->ws != nullptr ) (void) hipFree( l_pk->ws );
    (void) hipGetLastError();
  };
  int64_t l_total = 0;
  for( int l_op = 0; l_op < 2; l_op++ ) {
    if( !l_best.use[l_op] ) continue;
    l_pk->use[l_op] = true;
    // the copy as [C and rows][K], rows l_best.pitch elements apart
    std::vector< int64_t > l_sz, l_si, l_so;
    int64_t l_s = 1;
    for( std::size_t l_i = l_k[l_best.order].size(); l_i-- > 0; ) {
      int64_t const l_id = l_k[l_best.order][l_i].id;
      l_sz.push_back( sizes[l_id] );
      l_si.push_back( l_st[l_op][l_id] );
      l_so.push_back( l_s );
      l_s *= sizes[l_id];
    }
    l_s = l_best.pitch;
    for( std::size_t l_i = l_rows[l_op].size(); l_i-- > 0; ) {
      l_sz.push_back( l_rows[l_op][l_i].size );
      l_si.push_back( l_rows[l_op][l_i].s );
      l_so.push_back( l_s );
      l_s *= l_rows[l_op][l_i].size;
    }
    std::reverse( l_sz.begin(), l_sz.end() );
    std::reverse( l_si.begin(), l_si.end() );
    std::reverse( l_so.begin(), l_so.end() );
    if( plan_permute( (int64_t) l_sz.size(), l_sz.data(), l_si.data(), l_so.data(), dtype_left, ETIR_KTYPE_COPY,
                      l_pk->perm[l_op] ) != ETIR_SUCCESS ) {
      drop();
      return;
    }
    l_pk->offset[l_op] = l_total;
    l_total += ( l_s * l_esz + 255 ) / 256 * 256;
  }
  Loops const & l_lp = l_best.loops;
  std::size_t l_free = 0, l_device = 0;
  if(    hipMemGetInfo( &l_free, &l_device ) != hipSuccess
      // memory that a program is about to need stays free
      || 8 * std::size_t( l_total ) > l_free
      || plan_contraction_impl( (int64_t) l_lp.type.size(), l_lp.type.data(), l_lp.size.data(), l_lp.s[0].data(),
                                l_lp.s[1].data(), l_lp.aux.data(), l_lp.out.data(), dtype_left, dtype_right,
                                dtype_comp, dtype_out, ktype_first_touch, ktype_main, ktype_last_touch, allow_split,
                                l_pk->cont, nullptr, false, true ) != ETIR_SUCCESS
      || hipMalloc( &l_pk->ws, (std::size_t) l_total ) != hipSuccess
      // the padding's zeros are there when this returns: the fill runs on the
      // null stream, which a non-blocking stream's first execution does not
      // wait for, and hipMemset may return before it has run
      || (    l_best.pitch != plan.K
           && (    hipMemset( l_pk->ws, 0, (std::size_t) l_total ) != hipSuccess
                || hipStreamSynchronize( nullptr ) != hipSuccess ) ) ) {
    drop();
    return;
  }
  plan.packed = l_pk;
  ContractionPlan const & l_in = l_pk->cont.partial ? *l_pk->cont.partial : l_pk->cont;
  plan.desc += std::string( " | packed" ) + ( l_best.use[0] ? " left" : "" ) + ( l_best.use[1] ? " right" : "" )
             + ": " + tile_str( l_in.tile ) + " K=" + std::to_string( l_best.pitch ) + " "
             + mode_str( l_in.mode_a ) + " " + mode_str( l_in.mode_b )
             + ( l_in.args.k_one_step ? " one_step" : "" )
             + ( l_in.args.out_run > 0 ? " runs=" + std::to_string( l_in.args.out_run ) : std::string() )
             + ( l_pk->cont.split > 1 ? " S=" + std::to_string( l_pk->cont.split ) : std::string() );
}

}  // namespace

int plan_contraction( int64_t            num_loops,
                      int32_t const    * dim_types,
                      int64_t const    * sizes,
                      int64_t const    * strides_left,
                      int64_t const    * strides_right,
                      int64_t const    * strides_out_aux,
                      int64_t const    * strides_out,
                      int32_t            dtype_left,
                      int32_t            dtype_right,
                      int32_t            dtype_comp,
                      int32_t            dtype_out,
                      int32_t            ktype_first_touch,
                      int32_t            ktype_main,
                      int32_t            ktype_last_touch,
                      ContractionPlan  & plan,
                      DevicePlacement  * place ) {
  bool const l_split = std::getenv( "ETIR_NO_SPLIT_K" ) == nullptr;
  int l_err = plan_contraction_impl( num_loops, dim_types, sizes, strides_left, strides_right, strides_out_aux,
                                     strides_out, dtype_left, dtype_right, dtype_comp, dtype_out,
                                     ktype_first_touch, ktype_main, ktype_last_touch, l_split, plan, place );
  // the allocation-free entry point has no memory for copies
  if( l_err == ETIR_SUCCESS && place == nullptr ) {
    try_pack( num_loops, dim_types, sizes, strides_left, strides_right, strides_out_aux, strides_out, dtype_left,
              dtype_right, dtype_comp, dtype_out, ktype_first_touch, ktype_main, ktype_last_touch, l_split, plan );
    if( plan.packed || plan.split > 1 ) {
      plan.order = std::make_shared< ExecOrder >();
      ETIR_HIP_CHECK( hipEventCreateWithFlags( &plan.order->done, hipEventDisableTiming ) );
    }
  }
  return l_err;
}

void release_contraction( ContractionPlan & plan ) {
  if( !plan.placed && plan.d_tables != nullptr ) (void) hipFree( plan.d_tables );
  if( !plan.placed && plan.d_ws != nullptr ) (void) hipFree( plan.d_ws );
  plan.d_tables = nullptr;
  plan.d_ws = nullptr;
  if( plan.partial ) {
    release_contraction( *plan.partial );
    plan.partial.reset();
  }
  if( plan.packed ) {
    release_contraction( plan.packed->cont );
    for( PermutePlan & l_p : plan.packed->perm ) release_permute( l_p );
    if( plan.packed->ws != nullptr ) (void) hipFree( plan.packed->ws );
    plan.packed.reset();
  }
  if( plan.order ) {
    if( plan.order->done != nullptr ) (void) hipEventDestroy( plan.order->done );
    plan.order.reset();
  }
}

static int enqueue( ContractionPlan const & plan,
                    void const            * left,
                    void const            * right,
                    void const            * out_aux,
                    void                  * out,
                    hipStream_t             stream );

// the packed form of a contraction
static int enqueue_packed( PackedContraction const & pk,
                           void const              * left,
                           void const              * right,
                           void const              * out_aux,
                           void                    * out,
                           hipStream_t               stream ) {
  void const * l_op[2] = { left, right };
  for( int l_i = 0; l_i < 2; l_i++ ) {
    if( !pk.use[l_i] ) continue;
    void * l_copy = static_cast< char * >( pk.ws ) + pk.offset[l_i];
    int l_err = launch_permute( pk.perm[l_i], l_op[l_i], l_copy, stream );
    if( l_err != ETIR_SUCCESS ) return l_err;
    l_op[l_i] = l_copy;
  }
  return enqueue( pk.cont, l_op[0], l_op[1], out_aux, out, stream );
}

int launch_contraction( ContractionPlan const & plan,
                        void const            * left,
                        void const            * right,
                        void const            * out_aux,
                        void                  * out,
                        hipStream_t             stream,
                        bool                    ordered ) {
  if( plan.C == 0 || plan.M == 0 || plan.N == 0 ) return ETIR_SUCCESS;
  if( out == nullptr || ( plan.K > 0 && ( left == nullptr || right == nullptr ) ) ) {
    return fail( ETIR_NO_DATA_PTR_PROVIDED, "contraction: null tensor pointer" );
  }
  if( plan.needs_aux && out_aux == nullptr ) {
    return fail( ETIR_NO_DATA_PTR_PROVIDED, "contraction: touch kernel needs the auxiliary tensor" );
  }
  if( !plan.order ) return enqueue( plan, left, right, out_aux, out, stream );
  if( stream != nullptr ) {
    // under stream capture the operands are read in place: replays of a graph
    // are ordered with nothing that uses the copies outside it
    hipStreamCaptureStatus l_cap = hipStreamCaptureStatusNone;
    hipError_t const l_he = hipStreamIsCapturing( stream, &l_cap );
    if( l_he != hipSuccess ) (void) hipGetLastError();
    if( l_he != hipSuccess || l_cap != hipStreamCaptureStatusNone ) {
      return enqueue( plan, left, right, out_aux, out, stream );
    }
  }
  auto go = [&]() {
    return plan.packed ? enqueue_packed( *plan.packed, left, right, out_aux, out, stream )
                       : enqueue( plan, left, right, out_aux, out, stream );
  };
  if( ordered ) return go();
  ExecOrder & l_o = *plan.order;
  std::lock_guard< std::mutex > l_guard( l_o.lock );
  if( !l_o.events && stream != nullptr ) {
    // the first execution outside the null stream: those before were on it
    if( l_o.ran ) ETIR_HIP_CHECK( hipEventRecord( l_o.done, nullptr ) );
    l_o.events = true;
  }
  // also where the stream handle is the last execution's, which costs nothing:
  // a handle names another stream once the first has been destroyed (its work
  // may still run) or, for the per-thread default stream, in another thread
  if( l_o.events && l_o.ran ) ETIR_HIP_CHECK( hipStreamWaitEvent( stream, l_o.done, 0 ) );
  int const l_err = go();
  // also after an error: what was enqueued still uses the plan's memory
  l_o.ran = true;
  if( l_o.events ) ETIR_HIP_CHECK( hipEventRecord( l_o.done, stream ) );
  return l_err;
}

// The kernels of one execution, operands read in place.
static int enqueue( ContractionPlan const & plan,
                    void const            * left,
                    void const            * right,
                    void const            * out_aux,
                    void                  * out,
                    hipStream_t             stream ) {
  if( plan.split > 1 ) {
    int l_err = enqueue( *plan.partial, left, right, nullptr, plan.d_ws, stream );
    if( l_err != ETIR_SUCCESS ) return l_err;
    ContractArgs const & p = plan.partial->args;
    SplitReduceArgs r{};
    r.ws = reinterpret_cast< float const * >( plan.d_ws );
    r.aux = plan.needs_aux ? out_aux : nullptr;
    r.out = out;
    r.tc_out = p.tc_out;              // the first C entries belong to split 0
    r.tc_aux = p.tc_aux;
    r.tm_out = p.tm_out;
    r.tm_aux = p.tm_aux;
    r.tn_out = p.tn_out;
    r.tn_aux = p.tn_aux;
    r.span = plan.out_span;
    r.n_flat = plan.out_dense;
    r.flat_aux = plan.out_dense_aux;
    r.flat_vec = ( r.n_flat > 0 && r.span % 4 == 0
                   && reinterpret_cast< uintptr_t >( out ) % uintptr_t( plan.dtype_out == ETIR_BF16 ? 8 : 16 ) == 0 ) ? 1 : 0;
    r.C = (int32_t) plan.C;
    r.M = p.M;
    r.N = p.N;
    r.S = plan.split;
    r.first_touch = plan.first_touch;
    r.last_touch = plan.last_touch;
    r.out_bf16 = ( plan.dtype_out == ETIR_BF16 ) ? 1 : 0;
    l_err = launch_split_reduce( r, stream );
    if( l_err != ETIR_SUCCESS ) return l_err;
    hipError_t l_he = hipGetLastError();
    if( l_he != hipSuccess ) {
      return fail( ETIR_UNDEFINED_ERROR, std::string( "split reduce launch failed: " ) + hipGetErrorString( l_he ) );
    }
    return ETIR_SUCCESS;
  }
  ContractArgs a = plan.args;
  a.a   = plan.swapped ? right : left;
  a.b   = plan.swapped ? left : right;
  a.aux = plan.needs_aux ? out_aux : nullptr;
  a.out = out;

  if( uintptr_t( out ) % 16 != 0 ) {
    a.out_v8 = 0;
    if( a.out_run > 0 ) {
      a.out_run = 0;
      a.tiles_n = (int32_t) ( ( plan.N + 127 ) / 128 );
    }
  }
  // vector paths need aligned base pointers; otherwise fall back to gathers
  int32_t l_ma = plan.mode_a;
  int32_t l_mb = plan.mode_b;
  int64_t const l_esz = ( plan.dtype_in == ETIR_BF16 ) ? 2 : ( plan.dtype_in == ETIR_FP64 ? 8 : 4 );
  auto align_of = [&]( int32_t mode ) -> uintptr_t {
    if( mode == LOAD_VEC_K || mode == LOAD_VEC_MN ) return 16;
    if( mode == LOAD_VEC8_K || mode == LOAD_VEC8_MN ) return 8;
    return uintptr_t( l_esz );
  };
  if( uintptr_t( a.a ) % align_of( l_ma ) != 0 ) l_ma = LOAD_SCALAR;
  if( uintptr_t( a.b ) % align_of( l_mb ) != 0 ) l_mb = LOAD_SCALAR;
  int32_t l_dma_variant = plan.dma_variant;
  int32_t l_tile = plan.tile;
  if(    ( l_tile == TILE_BF16_DMA_256x256 || l_tile == TILE_BF16_DMA_256x128 || l_tile == TILE_F32_KWAVE_32x32
           || l_tile == TILE_F32_DMA_128x128 || l_tile == TILE_BF16_DMA_128x128
           || l_tile == TILE_F64_DMA_128x128 )
      && ( l_ma != plan.mode_a || l_mb != plan.mode_b ) ) {
    // the DMA and K-over-waves kernels need the 16-byte vector modes: use
    // the register-staged kernel with its own tile grid
    l_tile = plan.tile_fallback;
    int64_t l_bm, l_bn;
    tile_shape( l_tile, l_bm, l_bn );
    a.tiles_m = (int32_t) ( ( plan.M + l_bm - 1 ) / l_bm );
    a.tiles_n = (int32_t) ( ( plan.N + l_bn - 1 ) / l_bn );
  }

  int64_t const l_grid = int64_t( a.tiles_m ) * a.tiles_n * a.C;
  if( l_grid > 0x7fffffffLL ) {
    return fail( ETIR_UNDEFINED_ERROR, "contraction: grid too large" );
  }
  bool const l_kaff = ( a.k_affine != 0 );
  uint32_t const l_g = (uint32_t) l_grid;
  int l_err;
  switch( l_tile ) {
    case TILE_F32_128x128:
    case TILE_F32_64x64:
    case TILE_BF16_256x256:
    case TILE_BF16_256x128:
    case TILE_BF16_128x128:
    case TILE_BF16_64x64:
      l_err = launch_contract_tile( l_tile, l_ma, l_mb, l_kaff, a, l_g, stream );
      break;
    case TILE_F64_DMA_128x128: l_err = launch_contract_f64_dma( a, l_g, stream ); break;
    case TILE_F64_64x64:    l_err = launch_contract_f64_64x64( l_ma, l_mb, l_kaff, a, l_g, stream ); break;
    case TILE_CPX_F32_64x64: l_err = launch_contract_cpx( false, l_ma, l_mb, l_kaff, a, l_g, stream ); break;
    case TILE_CPX_F64_64x64: l_err = launch_contract_cpx( true, l_ma, l_mb, l_kaff, a, l_g, stream ); break;
    case TILE_F32_KWAVE_32x32:
      l_err = launch_contract_kwave( plan.kwave_waves, plan.kwave_kw, a, l_g, stream );
      break;
    case TILE_BF16_DMA_256x256:
      l_err = launch_contract_bf16_dma( l_ma, l_mb, l_dma_variant, a, l_g, stream );
      break;
    case TILE_BF16_DMA_256x128:
      l_err = launch_contract_bf16_dma( l_ma, l_mb, 2, a, l_g, stream );
      break;
    case TILE_BF16_DMA_128x128:
      l_err = launch_contract_bf16_dma( l_ma, l_mb, 4, a, l_g, stream );
      break;
    case TILE_F32_DMA_128x128:
      l_err = launch_contract_f32_dma( l_ma, l_mb, a, l_g, stream );
      break;
    case TILE_GEMV:
      l_err = launch_contract_gemv( plan.dtype_in == ETIR_BF16, a, stream );
      break;
    case TILE_SKINNY:
      l_err = launch_contract_skinny( plan.dtype_in == ETIR_BF16, a, stream );
      break;
    case TILE_PANEL:
      l_err = launch_contract_panel( a, stream );
      break;
    default: return fail( ETIR_COMPILATION_FAILED, "contraction: unknown tile configuration" );
  }
  if( l_err != ETIR_SUCCESS ) return l_err;
  hipError_t l_he = hipGetLastError();
  if( l_he != hipSuccess ) {
    return fail( ETIR_UNDEFINED_ERROR, std::string( "contraction launch failed: " ) + hipGetErrorString( l_he ) );
  }
  return ETIR_SUCCESS;
}

}  // namespace etir
