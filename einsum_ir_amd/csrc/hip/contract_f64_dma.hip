// fp64 contraction kernel with direct-to-LDS operand loads, both operands
// K-contiguous:
//   out[c][m][n] = touch( sum_k A[c][m][k] * B[c][n][k] )
// (reference src/basic/binary/ContractionBackendTpp.cpp:127-163 for the touch
// kernels), 128 x 128 tiles, k step 16, 8 waves of 32 x 64
// (v_mfma_f64_16x16x4_f64), two LDS stages of 32 KB (two workgroups per CU).
//
// MFMA-bound: a step's MFMAs take 4096 clocks per CU, its operands one
// direct-to-LDS load of 32 KB.  The 64 x 64 register-staged tile reads each
// operand twice as often and stages it through registers and ds_write between
// the MFMAs of one step: mk,nk->mn 2048 a side 335 us (51 TFLOP/s).
//
// LDS: [R][16] doubles, 128 bytes a row, the 16-byte segment g (2 k) of row r
// stored at g ^ swz_k(r), the byte layout of the fp32 kernel's K-contiguous
// stage.  A fragment read (8 bytes: row lane % 16, k 4 s + lane / 16) of half a
// wave covers 16 rows x 16 bytes, which the swizzle puts in 64 banks.
#include "contract_dma.h"

namespace etir {
namespace kern {

typedef double f64x4 __attribute__( ( ext_vector_type( 4 ) ) );

// 128 rows of one operand: 16 KiB-chunks over 8 waves, 8 rows a chunk
struct F64DmaLoader {
  static constexpr int NJ = 2;
  uint32_t m_off[NJ];   // byte offset of the lane's segment at k step 0 (kDmaOob: row outside)
  int32_t  m_kl[NJ];    // first k of the lane's segment within the step

  __device__ inline void init( int32_t const * tab_rows, int32_t rows, int32_t row0, int wave, int lane ) {
#pragma unroll
    for( int l_j = 0; l_j < NJ; l_j++ ) {
      int const l_r = ( wave * NJ + l_j ) * 8 + lane / 8;
      int const l_g = ( lane % 8 ) ^ int( swz_k( l_r ) );
      int32_t const l_row = row0 + l_r;
      m_kl[l_j]  = 2 * l_g;
      m_off[l_j] = ( l_row < rows ) ? uint32_t( 8 * ( tab_rows[l_row] + 2 * l_g ) ) : kDmaOob;
    }
  }
  // loads of step k0 (bytes kb past step 0); segments at or past K read zeros
  __device__ __attribute__( ( always_inline ) ) inline void issue( i32x4 rsrc, uint32_t lds_stage, int wave,
                                                                   int32_t k0, int32_t K, uint32_t kb ) {
#pragma unroll
    for( int l_j = 0; l_j < NJ; l_j++ ) {
      uint32_t const l_off = ( k0 + m_kl[l_j] < K ) ? m_off[l_j] + kb : kDmaOob;
      dma16( rsrc, l_off, lds_stage + ( wave * NJ + l_j ) * 1024 );
    }
  }
};

__global__ __launch_bounds__( 512, 2 )
void contract_f64_dma_kernel( ContractArgs a ) {
  constexpr int BM = 128, BN = 128, BK = 16;
  constexpr int SA = BM * BK * 8;                 // bytes of one operand's stage
  __shared__ __attribute__( ( aligned( 1024 ) ) ) char l_lds[4 * SA];

  int32_t const l_nblk = gridDim.x;
  int32_t l_bid = blockIdx.x;
  if( ( l_nblk & 7 ) == 0 ) l_bid = ( l_bid & 7 ) * ( l_nblk >> 3 ) + ( l_bid >> 3 );
  int32_t l_c, l_m0, l_n0;
  decode_tile< BM, BN >( a, l_bid, l_c, l_m0, l_n0 );

  int const l_lane = threadIdx.x & 63;
  int const l_wave = __builtin_amdgcn_readfirstlane( threadIdx.x >> 6 );
  int const l_wm   = l_wave >> 1;
  int const l_wn   = l_wave & 1;
  int const l_r16  = l_lane & 15;
  int const l_k4   = l_lane >> 4;

  i32x4 const l_ra = make_rsrc( reinterpret_cast< double const * >( a.a ) + a.tc_a[l_c], kDmaOob );
  i32x4 const l_rb = make_rsrc( reinterpret_cast< double const * >( a.b ) + a.tc_b[l_c], kDmaOob );
  F64DmaLoader l_lda, l_ldb;
  l_lda.init( a.tm_a, a.M, l_m0, l_wave, l_lane );
  l_ldb.init( a.tn_b, a.N, l_n0, l_wave, l_lane );

  // output offsets of this lane's rows and columns (clamped), read here so
  // that the epilogue's stores wait for no load
  int32_t l_mo[2][4], l_no[4];
#pragma unroll
  for( int l_i = 0; l_i < 2; l_i++ )
#pragma unroll
    for( int l_r = 0; l_r < 4; l_r++ )
      l_mo[l_i][l_r] = a.tm_out[min( l_m0 + l_wm * 32 + l_i * 16 + 4 * l_r + l_k4, a.M - 1 )];
#pragma unroll
  for( int l_j = 0; l_j < 4; l_j++ ) l_no[l_j] = a.tn_out[min( l_n0 + l_wn * 64 + l_j * 16 + l_r16, a.N - 1 )];

  f64x4 l_acc[2][4];
#pragma unroll
  for( int l_i = 0; l_i < 2; l_i++ )
#pragma unroll
    for( int l_j = 0; l_j < 4; l_j++ ) l_acc[l_i][l_j] = f64x4( 0.0 );

  // byte of (row r16 of the wave's first block, k) in a stage: rows 16 apart
  // share the swizzle, so blocks are 16 rows of 128 bytes apart
  uint32_t l_seg[BK / 4];
#pragma unroll
  for( int l_s = 0; l_s < BK / 4; l_s++ ) {
    l_seg[l_s] = uint32_t( ( ( 2 * l_s + ( l_k4 >> 1 ) ) ^ int( swz_k( l_r16 ) ) ) * 16 + ( l_k4 & 1 ) * 8 );
  }
  uint32_t const l_pa = uint32_t( ( l_wm * 32 + l_r16 ) * 128 );
  uint32_t const l_pb = uint32_t( SA + ( l_wn * 64 + l_r16 ) * 128 );

  int32_t const  l_nk   = ( a.K + BK - 1 ) / BK;
  uint32_t const l_lds0 = lds_addr( l_lds );
  if( l_nk > 0 ) {
    l_lda.issue( l_ra, l_lds0, l_wave, 0, a.K, 0u );
    l_ldb.issue( l_rb, l_lds0 + SA, l_wave, 0, a.K, 0u );
    wait_vmcnt< 0 >();
    barrier_lds();
    for( int32_t l_kt = 0; l_kt < l_nk; l_kt++ ) {
      char const * l_st = l_lds + ( l_kt & 1 ) * 2 * SA;
      // the other stage was last read in the step before, which ended with a
      // barrier; loads of the step past the last read zeros
      uint32_t const l_nst = l_lds0 + uint32_t( ( l_kt & 1 ) ^ 1 ) * 2 * SA;
      l_lda.issue( l_ra, l_nst, l_wave, ( l_kt + 1 ) * BK, a.K, uint32_t( l_kt + 1 ) * BK * 8 );
      l_ldb.issue( l_rb, l_nst + SA, l_wave, ( l_kt + 1 ) * BK, a.K, uint32_t( l_kt + 1 ) * BK * 8 );
#pragma unroll
      for( int l_s = 0; l_s < BK / 4; l_s++ ) {
        double l_fa[2], l_fb[4];
#pragma unroll
        for( int l_i = 0; l_i < 2; l_i++ )
          l_fa[l_i] = *reinterpret_cast< double const * >( l_st + l_pa + l_seg[l_s] + l_i * 16 * 128 );
#pragma unroll
        for( int l_j = 0; l_j < 4; l_j++ )
          l_fb[l_j] = *reinterpret_cast< double const * >( l_st + l_pb + l_seg[l_s] + l_j * 16 * 128 );
#pragma unroll
        for( int l_i = 0; l_i < 2; l_i++ )
#pragma unroll
          for( int l_j = 0; l_j < 4; l_j++ )
            l_acc[l_i][l_j] = __builtin_amdgcn_mfma_f64_16x16x4f64( l_fa[l_i], l_fb[l_j], l_acc[l_i][l_j], 0, 0, 0 );
      }
      // the next stage has landed (own loads: vmcnt; everyone's: barrier) and
      // every wave is done reading this one
      wait_vmcnt< 0 >();
      wait_lgkmcnt0();
      barrier_lds();
    }
  }

  // epilogue: touch kernels per element, 16 consecutive columns per 16 lanes
  double * l_out = reinterpret_cast< double * >( a.out ) + a.tc_out[l_c];
  double const * l_aux = reinterpret_cast< double const * >( a.aux ) + ( a.aux != nullptr ? a.tc_aux[l_c] : 0 );
  bool const l_read_out  = ( a.first_touch == ETIR_KTYPE_ADD || a.first_touch == ETIR_KTYPE_UNDEFINED );
  bool const l_aux_first = ( a.first_touch == ETIR_KTYPE_ADD || a.first_touch == ETIR_KTYPE_COPY );
  bool const l_aux_last  = ( a.last_touch == ETIR_KTYPE_ADD );
  bool const l_relu      = ( a.last_touch == ETIR_KTYPE_RELU );
#pragma unroll
  for( int l_i = 0; l_i < 2; l_i++ ) {
#pragma unroll
    for( int l_r = 0; l_r < 4; l_r++ ) {
      int32_t const l_m = l_m0 + l_wm * 32 + l_i * 16 + 4 * l_r + l_k4;
      if( l_m >= a.M ) continue;
      int32_t const l_ma = ( l_aux_first || l_aux_last ) ? a.tm_aux[l_m] : 0;
#pragma unroll
      for( int l_j = 0; l_j < 4; l_j++ ) {
        int32_t const l_n = l_n0 + l_wn * 64 + l_j * 16 + l_r16;
        if( l_n >= a.N ) continue;
        int64_t const l_off = int64_t( l_mo[l_i][l_r] ) + l_no[l_j];
        double l_v = l_acc[l_i][l_j][l_r];
        double l_x = 0.0;
        if( l_aux_first || l_aux_last ) l_x = l_aux[ int64_t( l_ma ) + a.tn_aux[l_n] ];
        if( l_read_out ) l_v = l_out[l_off] + l_v;
        if( l_aux_first ) l_v = l_x + l_v;
        if( l_relu ) l_v = fmax( l_v, 0.0 );
        else if( l_aux_last ) l_v = l_v + l_x;
        l_out[l_off] = l_v;
      }
    }
  }
}

}  // namespace kern

int launch_contract_f64_dma( ContractArgs const & a, uint32_t grid, hipStream_t stream ) {
  hipLaunchKernelGGL( kern::contract_f64_dma_kernel, dim3( grid ), dim3( 512 ), 0, stream, a );
  return ETIR_SUCCESS;
}

}  // namespace etir
