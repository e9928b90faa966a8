#include <hip/hip_runtime.h>
#include "mfma_rows.h"
#include <cstdio>
#include <cstdlib>
#include <vector>
#include <algorithm>
using namespace xllm;
#define CK(x) do{hipError_t e=(x); if(e!=hipSuccess){printf("err %s line %d\n",hipGetErrorString(e),__LINE__);exit(1);}}while(0)
// MODE 0: global_load_lds rows of 256 B (4 per instr), stride; 1: buffer lds; 2: VGPR loads rows of 256 B; 3: VGPR 16 rows x 64 B; 4: contiguous 1 KB lds ; 5: 8 rows x 128 B lds
// region: rows x stride bytes ; each wave walks columns of its 16 rows
template<int MODE,int DEPTH> __global__ __launch_bounds__(256) void k(const char* p, float* out, int iters, int stride, int rows, int cols, int nrow0){
  __shared__ __attribute__((aligned(1024))) unsigned short lds[4*8192];
  int lane=threadIdx.x&63, wid=__builtin_amdgcn_readfirstlane(threadIdx.x>>6);
  unsigned short* dst=lds+wid*8192;
  int r0=((blockIdx.x*64+wid*16)%rows);
  const char* base=p+(long)r0*stride;
  unsigned o[4];
  for(int i=0;i<4;i++){
    if(MODE==0||MODE==1||MODE==2) o[i]=(i*4+(lane>>4))*stride+(lane&15)*16;
    if(MODE==3) o[i]=(lane&15)*stride+(lane>>4)*16+i*64;
    if(MODE==4) o[i]=i*1024+lane*16;
    if(MODE==5) o[i]=((i>>1)*8+(lane>>3))*stride+(lane&7)*16+(i&1)*128;
  }
  unsigned long long acc=0;
  auto rs=mr_buffer(base,(unsigned)(16*stride));
  uint4 v[DEPTH][4];
  for(int t=0;t<iters;t+=DEPTH){
#pragma unroll
    for(int d=0;d<DEPTH;d++){
      int c=((t+d)%cols)*(MODE==4?4096:256);
#pragma unroll
      for(int i=0;i<4;i++){
        if(MODE==0||MODE==4||MODE==5) __builtin_amdgcn_global_load_lds((glb_void*)(base+c+o[i]),(lds_void*)(dst+((d%4)*4+i)*512),16,0,0);
        else if(MODE==1) mr_to_lds(rs,o[i]+c,dst+((d%4)*4+i)*512);
        else v[d][i]=*(const uint4*)(base+c+o[i]);
      }
    }
    if(MODE==2||MODE==3){
#pragma unroll
      for(int d=0;d<DEPTH;d++) for(int i=0;i<4;i++){acc+=v[d][i].x^v[d][i].y^v[d][i].z^v[d][i].w;}
    } else asm volatile("s_waitcnt vmcnt(0)":::"memory");
  }
  if(out && acc==123456789ull) out[0]=1;
}
template<int MODE,int DEPTH> void go(const char*name,const char*p,int stride,int rows,int cols){
  int iters=512; hipEvent_t a,b;CK(hipEventCreate(&a));CK(hipEventCreate(&b)); std::vector<float> ts;
  for(int r=0;r<5;r++){CK(hipEventRecord(a));k<MODE,DEPTH><<<256,256>>>(p,nullptr,iters,stride,rows,cols,0);CK(hipEventRecord(b));CK(hipEventSynchronize(b));float ms;CK(hipEventElapsedTime(&ms,a,b));ts.push_back(ms*1000);}
  CK(hipGetLastError());
  std::sort(ts.begin(),ts.end()); double bytes=(double)iters*4*4096; printf("%s depth %d stride %d rows %d cols %d: %.1f us  %.1f KB/us/CU\n",name,DEPTH,stride,rows,cols,ts[1],bytes/1024/ts[1]);fflush(stdout);
}
int main(){
  char*p;CK(hipMalloc(&p,256<<20));CK(hipMemset(p,1,256<<20));CK(hipDeviceSynchronize());
  // 512 rows x 4096 B = 2 MB: in each XCD's L2
  go<0,4>("lds 4x256",p,4096,512,16); go<0,8>("lds 4x256",p,4096,512,16);
  go<1,4>("buf 4x256",p,4096,512,16); go<1,8>("buf 4x256",p,4096,512,16);
  go<4,8>("lds 1KB  ",p,65536,32,16); go<5,8>("lds 8x128",p,4096,512,16);
  go<2,4>("reg 4x256",p,4096,512,16); go<2,8>("reg 4x256",p,4096,512,16); go<3,8>("reg 16x64",p,4096,512,16);
  go<0,8>("lds 4x256 odd",p,4096+256,480,16); go<2,8>("reg 4x256 odd",p,4096+256,480,16);
  go<0,8>("lds 4x256 16 rows (L1/L2 hot)",p,4096,64,4);
  return 0;
}
